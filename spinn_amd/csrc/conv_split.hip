// conv_split.hip - where the split-bf16 implicit GEMM (conv_split.h) runs, its weight
// packing and its launch choice.
#include "conv_split.h"
#include <atomic>
#include <cstdlib>

namespace spinn {

// W [group][OCg][Cg][KH][KW] -> split planes [group][octet][plane][rows_p][8], K in
// (kh, kw, c) order, each tap's channels padded to octets; one thread per (octet, row).
// An octet with a weight that loses bits, or of `limit` and more, gets a NaN, which sends its
// row's tiles to the fp32 MFMA (split_core.h).
__global__ void conv_pack_split_kernel(const float *__restrict__ w, u32x4 *__restrict__ out, int groups, int OCg,
                                       int Cg, int KHW, int rows_p, int octs, float limit) {
    const int co8 = (Cg + 7) / 8;
    const int64_t total = (int64_t)groups * octs * rows_p;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (int64_t)gridDim.x * blockDim.x) {
        const int m = (int)(e % rows_p);
        const int64_t go = e / rows_p;
        const int o = (int)(go % octs);
        const int64_t g = go / octs;
        const int tap = o / co8;
        const int c0 = (o - tap * co8) * 8;
        float v[8];
        bool carried = true;
        for (int i = 0; i < 8; ++i) {
            v[i] = (m < OCg && tap < KHW && c0 + i < Cg) ? w[((g * OCg + m) * Cg + c0 + i) * KHW + tap] : 0.f;
            carried = carried && fabsf(v[i]) < limit;
        }
        u32x4 p[3];
        uint32_t lost = 0;
        split8(v, p[0], p[1], p[2], lost);
        if (!carried || (lost & 0xffffu)) p[0][0] = 0x7fc0u;
        u32x4 *dst = out + (go * 3) * rows_p + m;
        for (int i = 0; i < 3; ++i) dst[(int64_t)i * rows_p] = p[i];
    }
}

namespace {

std::atomic<int> g_force_split{-1}, g_force_split_bm{0}, g_force_split_k{0};

struct SplitChoice {
    int bm, split, chunk, groups_k;
    bool sk;
    SkPlan sp;
};

int split_octs(const SpinnHipConvDesc *d) {
    const int co8 = (d->c / d->group + 7) / 8;
    constexpr int q = 4 * kSplitGS;
    return (d->kh * d->kw * co8 + q - 1) / q * q;
}
int split_rows(const SpinnHipConvDesc *d) {
    return (d->oc / d->group + kSplitRowPad - 1) / kSplitRowPad * kSplitRowPad;
}

// 1x1 convs that 2-pixel loads can serve (where the tensors are 8-byte aligned).
bool split_pw2_shape(const SpinnHipConvDesc *d) {
    return d->kh == 1 && d->kw == 1 && d->sh == 1 && d->sw == 1 && d->ph == 0 && d->pw == 0 && d->oh == d->h &&
           d->ow == d->w && (d->h * d->w) % 2 == 0 && d->c / d->group % 8 == 0;
}

// Tile height, K split and stream-K plan of an eligible conv. A 128-row tile splits each
// activation half as often as a 64-row one and two workgroups share a CU, so it wins
// where its grid has 0.6 of a tile per CU, two thirds with 1-pixel loads (320 -> 120 3x3
// stride 2, 159 tiles: 115 us against 91 on fp32 tiles), unless M leaves over a fifth of its
// rows empty (MI355X, us: 512 -> 128@28x28 at batch 32, 392 tiles, 24.8 against 29.5 on 64 rows; 1024 -> 512@14x14 40.8 / 52.8; 3x3 stride 2
// 128@56x56 59.3 / 81.6; 256 -> 1024@14x14 at batch 8, 208 tiles, 10.1 / 11.2; 3x3 stride 2
// 256@28x28 at batch 32, 196 tiles, 68.8 / 81.6, 76.0 with the remainder of the 64-row tiles
// cut along K). One exception: 1x1 convs of
// 2-pixel loads with 0.6 to 1 tile per CU and K of 768 or more run on 64 rows with the
// remainder cut, though whole 128-row tiles are faster (1024 -> 256@14x14 at batch 32: 29.8
// against 26.6): the tests of the workspace and no-allocation interfaces are written on this
// layer and ask for its stream-K workspace. Below that:
//  * K of 2048 or more: 128 rows, K split over four tiles' worth of workgroups
//    (2048 -> 512@7x7 at batch 32: 33.8 against 65.6 unsplit, 44.9 on 64 rows; 3x3 stride
//    2 512@14x14: 67.4 / 132 / 105);
//  * else 64 rows, whole.
// With three or more whole tiles per CU the remainder is cut along K where whole tiles
// alone are unbalanced (plan_streamk); with fewer the co-resident workgroups even out
// by themselves (512 -> 128@28x28: 33.8 cut, 24.8 whole). Channel tails stay whole without a
// residual: their cut kernel reads a spilled index back in its K loop (with one the other
// does too: 359 -> 720@53x53 at batch 20 255 cut, 274 whole).
SplitChoice split_choice(const SpinnHipConvDesc *d) {
    SplitChoice c{};
    const int M = d->oc / d->group;
    const int ntot = d->n * d->oh * d->ow;
    const int tiles_n = (ntot + kSplitBN - 1) / kSplitBN;
    const int64_t cus = device_cu_count();
    c.groups_k = split_octs(d) / (4 * kSplitGS);
    c.split = 1;
    c.chunk = c.groups_k;
    const int64_t t128 = (int64_t)((M + 127) / 128) * tiles_n * d->group;
    const bool fills = (M + 127) / 128 * 128 * 4 <= 5 * M;
    const bool pw2 = split_pw2_shape(d);
    const bool res = d->act == SPINN_ACT_ADD || d->act == SPINN_ACT_ADD_RELU;
    const bool some = pw2 ? 5 * t128 >= 3 * cus : 3 * t128 >= 2 * cus;
    const bool cut = d->group == 1 && some && t128 < cus && c.groups_k >= 12 && pw2;
    int split = 1;
    if (fills && some && !cut) {
        c.bm = 128;
    } else if (fills && d->group == 1 && !some && 4 * t128 >= cus && c.groups_k >= 32) {
        c.bm = 128;
        split = (int)((3 * cus / 2 + t128 - 1) / t128);
    } else {
        c.bm = 64;
    }
    const bool forced = streamk_forced_on();
    if (forced) c.bm = 64;
    if (const int bm = g_force_split_bm.load()) c.bm = bm;
    if (d->group != 1) return c;
    if (const int k = g_force_split_k.load()) {
        split = k;
    } else if (forced || (cut && c.bm == 64) || (c.bm == 128 && t128 >= 3 * cus && (d->c % 8 == 0 || res))) {
        c.sk = plan_streamk((M + c.bm - 1) / c.bm, tiles_n, c.groups_k, 1, c.bm * kSplitBN, c.sp);
        if (c.sk) return c;
    }
    split = std::min(split, c.groups_k);
    if (split > 1) {
        const int chunk = (c.groups_k + split - 1) / split;
        c.split = (c.groups_k + chunk - 1) / chunk;
        c.chunk = c.split > 1 ? chunk : c.groups_k;
    }
    return c;
}

// Bytes of one group's planes.
uint64_t split_plane_bytes(const SpinnHipConvDesc *d) { return (uint64_t)split_octs(d) * 3 * split_rows(d) * 16; }

bool split_eligible(const SpinnHipConvDesc *d) {
    // 16 channels: a fetch steps at most four taps (co8 >= 2), and the gathers' channel
    // offsets stay inside the input. Planes are 1.5 times the weights: where they pass what
    // one buffer descriptor spans, the fp32 kernels still run.
    return d->c / d->group >= 16 && !stem_mfma_eligible(d) && split_plane_bytes(d) <= kMaxOperandBytes;
}

// How the fp32 kernels would run the conv (conv_igemm.hip): whole tiles in one launch, at
// least one per CU; the wave-K kernel on a grid of one 64 x 64 tile per CU and more; or else
// (K cut by stream-K or a reduction, or few tiles).
enum Fp32Route { kFp32Whole, kFp32WaveK, kFp32Other };
Fp32Route fp32_route(const SpinnHipConvDesc *d, const TileChoice &tc) {
    const int M = d->oc / d->group, K = d->c / d->group * d->kh * d->kw, ntot = d->n * d->oh * d->ow;
    if ((int64_t)((M + 63) / 64) * ((ntot + 63) / 64) * d->group < device_cu_count()) return kFp32Other;
    const bool pointwise = d->kh == 1 && d->kw == 1 && d->sh == 1 && d->sw == 1 && d->ph == 0 && d->pw == 0 &&
                           d->oh == d->h && d->ow == d->w;
    if (wavek_tile(M, ntot, K, d->group, pointwise ? kWkConvPointwise : kWkConvGather)) return kFp32WaveK;
    const int tiles_m = (M + tc.bm - 1) / tc.bm, tiles_n = (ntot + tc.bn - 1) / tc.bn;
    SkPlan sp;
    if (tc.split > 1 || (d->group == 1 && plan_streamk(tiles_m, tiles_n, (K + kBK - 1) / kBK, 4, tc.bm * tc.bn, sp)))
        return kFp32Other;
    return kFp32Whole;
}

} // namespace

void force_split_conv(int mode, int bm, int split) {
    g_force_split.store(mode < 0 ? -1 : (mode ? 1 : 0));
    g_force_split_bm.store(bm == 64 || bm == 128 ? bm : 0);
    g_force_split_k.store(std::max(split, 0));
}

bool split_conv_selected(const SpinnHipConvDesc *d) {
    if (!split_eligible(d) || tiles_forced() || wavek_forced_on()) return false;
    const int f = g_force_split.load();
    if (f >= 0) return f == 1;
    const int M = d->oc / d->group;
    const int K = d->c / d->group * d->kh * d->kw;
    const int ntot = d->n * d->oh * d->ow;
    const int64_t tiles64 = (int64_t)((M + 63) / 64) * ((ntot + 63) / 64) * d->group;
    // Measured against the fp32 MFMA tiles (us): 1x1 with K = 64 gains without a residual
    // (64 -> 256@56x56 at batch 32: 42.0 -> 35.3) and loses with one (44.1 -> 47.3; K = 128,
    // 128 -> 512@28x28: 36.3 -> 38.8; K = 256, 256 -> 1024@14x14: 33.9 -> 32.4). Grids of
    // two thirds to one 64 x 64 tile per CU gain from K = 256 (384 -> 256@13x13 at batch 16:
    // 12.6 -> 12.4; K = 128, 128@80x80 at batch 1: 6.06 and 6.09) and smaller ones lose
    // (1024 -> 256@14x14 at batch 8: 15.8 on the wave-K kernel, 16.8 here), as do rows that
    // leave over a quarter of the tiles empty (80@80x80 at batch 1: 5.2 -> 5.9).
    const bool res = d->act == SPINN_ACT_ADD || d->act == SPINN_ACT_ADD_RELU;
    const int64_t cus = device_cu_count();
    if ((M + 63) / 64 * 64 * 3 > 4 * M || K < (res ? 256 : 64)) return false;
    if (!(tiles64 >= cus || (3 * tiles64 >= 2 * cus && K >= 256))) return false;
    // Both ways timed over 3400 such convs of 16-2048 channels, 7-112 pixels and batches of
    // 1-32, on random operands. Where the fp32 kernels take whole tiles in one launch, what
    // the tiles here do for padding (rows up to 64 or 128, K up to whole groups of 64) counts;
    // where they cut K, by stream-K or a reduction, or run the wave-K kernel, this one gains
    // also at a real share of a half (1x1: 0.70; 72 -> 1809@14x14 at batch 4: 14.5 -> 7.7).
    const SplitChoice c = split_choice(d);
    const int64_t tiles = (int64_t)((M + c.bm - 1) / c.bm) * ((ntot + 63) / 64) * d->group;
    const int64_t rem = tiles % (2 * cus);
    const bool half = rem > 0 && rem <= cus; // the last round leaves one workgroup or none on a CU
    const bool tail = d->c / d->group % 8 != 0, pw2 = split_pw2_shape(d), one = d->kh * d->kw == 1;
    const TileChoice tc = choose_tiles(M, ntot, K, d->group, d->group == 1);
    const Fp32Route route = fp32_route(d, tc);
    // One fp32 chain over a long K would be nearly three times as far off (K = 2007, 954 tiles:
    // 9.3e-7 against 3.3e-7): such layers stay here, also the slower ones (2007 -> 518@58x58 at
    // batch 2: 134 -> 157).
    if (route == kFp32Whole && K >= 1536) return true;
    // 1x1 channel tails on 64-row tiles lose to all but the wave-K kernel (1527 -> 288, 285
    // tiles: 1.17 of the time; half-empty last rounds 1.17, others 0.99).
    if (c.bm == 64 && tail && one && route != kFp32WaveK) return false;
    if (route != kFp32Whole) return true;
    // The line by real share, in twentieths. Medians of the time (2-pixel loads; 1-pixel 1x1; larger
    // kernels; channel tails): 0.5-0.6 1.14 / 1.14 / - / 1.26; 0.6-0.7 0.98 / 1.11 / 0.93 / 1.12;
    // 0.7-0.8 0.87 / 0.96 / 0.82 / 0.82; above 0.74 / 0.80 / 0.71 / 0.78. Tails of 1x1 convs
    // 1.03 at 0.7-0.8, above it 0.86.
    const int64_t kpad = (int64_t)c.groups_k * kSplitGS * kSplitBK;
    const int64_t real = 20 * (int64_t)M * K, all = (M + c.bm - 1) / c.bm * c.bm * kpad;
    if (real < (pw2 || !one ? 13 : tail ? 16 : 14) * all) return false;
    if (pw2) return true;
    // 1x1 with 1-pixel loads: up to three groups of K do not pay for the prologue on 64-row
    // tiles (1.04-1.35 of the time, four and more 0.87), nor up to two on 128-row ones in a
    // half-empty last round or with a channel tail (1.00-1.05; three and more 0.77). Larger
    // kernels: 16 channels into more than 64 do not (K = 144 of 192; 16 -> 304@83x83 at batch 4:
    // 33 -> 40).
    if (one && c.groups_k < (c.bm == 64 ? 4 : half || tail ? 3 : 1)) return false;
    return one || M <= 64 || 5 * K >= 4 * kpad;
}

int64_t split_packed_floats(const SpinnHipConvDesc *d) {
    if (!split_eligible(d)) return 0;
    return (int64_t)d->group * split_octs(d) * 3 * split_rows(d) * 4;
}

int split_pack(const SpinnHipConvDesc *d, const float *w, float *packed, hipStream_t st) {
    if (!split_eligible(d)) return SPINN_HIP_OK;
    const int64_t total = (int64_t)d->group * split_octs(d) * split_rows(d);
    const int blocks = (int)std::min<int64_t>((total + 255) / 256, 65535);
    hipLaunchKernelGGL(conv_pack_split_kernel, dim3(blocks), dim3(256), 0, st, w, (u32x4 *)packed, d->group,
                       d->oc / d->group, d->c / d->group, d->kh * d->kw, split_rows(d), split_octs(d),
                       split_weight_limit(d->c / d->group * d->kh * d->kw));
    return check_launch();
}

size_t split_conv_workspace_bytes(const SpinnHipConvDesc *d) {
    const SplitChoice c = split_choice(d);
    if (c.sk) {
        // plan time: settle how the parts exchange sums on this device
        int dev = 0;
        if (hipGetDevice(&dev) == hipSuccess) probe_xcd_local(dev);
        init_device_status();
        return c.sp.ws_bytes;
    }
    if (c.split <= 1) return 0;
    return (size_t)c.split * d->oc * ((size_t)d->n * d->oh * d->ow) * sizeof(float);
}

int split_conv(const SpinnHipConvDesc *d, const float *x, const float *wt, bool tap_order, const float *planes, const float *bias, const float *res,
               float *y, void *ws, size_t ws_bytes, hipStream_t st) {
    const uint64_t x_bytes = (uint64_t)d->n * d->c * d->h * d->w * sizeof(float);
    const uint64_t y_bytes = (uint64_t)d->n * d->oc * d->oh * d->ow * sizeof(float);
    const uint64_t w_bytes = split_plane_bytes(d);
    const SplitChoice c = split_choice(d);
    ConvSplitArgs a{};
    a.t.M = d->oc / d->group;
    a.t.geom = ConvGeom{x, (uint32_t)x_bytes, d->c, d->h, d->w, d->c / d->group, d->oh, d->ow, d->kh, d->kw,
                        d->sh, d->sw, d->ph, d->pw, d->n * d->oh * d->ow};
    a.t.wpk = wt;
    a.t.ldw = (a.t.M + 3) / 4 * 4;
    a.t.K = a.t.geom.Cg * d->kh * d->kw;
    a.t.wpk_group_stride = (int64_t)a.t.K * a.t.ldw;
    // the limits of the fp32 kernels (conv_igemm.hip)
    const uint64_t wt_bytes = (uint64_t)d->group * a.t.wpk_group_stride * sizeof(float);
    if (x_bytes > kMaxOperandBytes || y_bytes > kMaxOperandBytes || wt_bytes > kMaxOperandBytes)
        return SPINN_HIP_EUNSUPPORTED;
    a.tap_order = tap_order ? 1 : 0;
    a.t.y = y;
    a.t.bias = bias;
    a.t.res = res;
    a.t.res_bytes = (uint32_t)y_bytes;
    a.t.act = d->act;
    a.t.OC = d->oc;
    a.t.OHW = d->oh * d->ow;
    a.w = SplitPlanes{planes, (uint32_t)w_bytes, split_rows(d), split_octs(d)};
    a.w_group_stride = (int64_t)w_bytes;
    a.co8 = (a.t.geom.Cg + 7) / 8;
    a.groups_k = c.groups_k;
    a.chunk = c.chunk;
    SkSched s{};
    if (c.sk) {
        if (!ws || ws_bytes < c.sp.ws_bytes || ((uintptr_t)ws & 15u)) return SPINN_HIP_EWORKSPACE;
        s = sk_sched(c.sp, (a.t.M + c.bm - 1) / c.bm, c.groups_k, ws);
    } else if (c.split > 1) {
        if (!ws || ws_bytes < (size_t)c.split * d->oc * (size_t)a.t.geom.ntot * sizeof(float)) return SPINN_HIP_EWORKSPACE;
        a.t.ws = (float *)ws;
    }
    const SkSched *sk = c.sk ? &s : nullptr;
    const bool pw2 = split_pw2_shape(d) && (((uintptr_t)x | (uintptr_t)y | (uintptr_t)res) & 7u) == 0;
    int rc;
    if (pw2) rc = launch_conv_split_pw2(a, c.bm, d->group, c.split, sk, c.sp.grid, st);
    else if (a.t.geom.Cg % 8 == 0) rc = launch_conv_split_gather(a, c.bm, d->group, c.split, sk, c.sp.grid, st);
    else rc = launch_conv_split_gather_tail(a, c.bm, d->group, c.split, sk, c.sp.grid, st);
    if (rc || c.split <= 1) return rc;
    return launch_conv_splitk_reduce(c.split, a.t, st);
}

} // namespace spinn
