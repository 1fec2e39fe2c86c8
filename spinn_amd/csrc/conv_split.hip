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
// stride 2, 159 tiles: 115 against 91 on fp32 tiles) (MI355X, us: 512 -> 128@28x28 at batch 32, 392
// tiles, 24.8 against 29.5 on 64 rows; 1024 -> 512@14x14 40.8 / 52.8; 3x3 stride 2
// 128@56x56 59.3 / 81.6; 256 -> 1024@14x14 at batch 8, 208 tiles, 10.1 / 11.2; 3x3 stride 2
// 256@28x28 at batch 32, 196 tiles, 68.8 / 81.6, 76.0 with the remainder of the 64-row tiles
// cut along K), unless M leaves over a fifth of its rows empty. One exception: 1x1 convs of
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
// by themselves (512 -> 128@28x28: 33.8 cut, 24.8 whole).
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
    } else if (forced || (cut && c.bm == 64) || (c.bm == 128 && t128 >= 3 * cus)) {
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
    // (64 -> 256@56x56 at batch 32: 42.0 -> 34.4) and loses with one (44.1 -> 47.3; K = 128,
    // 128 -> 512@28x28: 36.3 -> 38.8; K = 256, 256 -> 1024@14x14: 33.9 -> 32.4). Grids of
    // two thirds to one 64 x 64 tile per CU gain from K = 256 (384 -> 256@13x13 at batch 16:
    // 12.6 -> 12.4; K = 128, 128@80x80 at batch 1: 6.06 and 6.09) and smaller ones lose
    // (1024 -> 256@14x14 at batch 8: 15.8 on the wave-K kernel, 16.8 here), as do rows that
    // leave over a quarter of the tiles empty (80@80x80 at batch 1: 5.2 -> 5.9).
    const bool res = d->act == SPINN_ACT_ADD || d->act == SPINN_ACT_ADD_RELU;
    const int64_t cus = device_cu_count();
    if ((M + 63) / 64 * 64 * 3 > 4 * M || K < (res ? 256 : 64)) return false;
    if (!(tiles64 >= cus || (3 * tiles64 >= 2 * cus && K >= 256))) return false;
    // What the tiles do for padding counts against their rate: rows up to 64 or 128, and K up
    // to whole groups of 64. Over 4000 shapes of 32-2048 channels, 7-112 pixels and batches of
    // 1-32, against the kernels they had (fp32 tiles, split K, wave-K), at a real share of
    //   under 0.7   0.93-1.19 of the time for 1x1 convs with 2-pixel loads, half of them
    //               slower (96 -> 2016@16x16: K = 96 in two groups, 1.4), above it 0.79;
    //   under 0.75  up to 1.47 for 1x1 convs with 1-pixel loads (64 -> 723@69x69 at batch 23:
    //               167 -> 246), above it 0.84; 3x3 ones gain down to 0.65, past 64
    //               rows to 0.7 (280 -> 88@55x55 at batch 17: 140 -> 173) and not with K under
    //               four fifths of its groups (16 -> 304@83x83 at batch 4: 33 -> 40);
    // and with 1-pixel loads one or two groups of K do not pay for their prologue (1.06).
    const SplitChoice c = split_choice(d);
    const int64_t rows = (M + c.bm - 1) / c.bm * c.bm, kpad = (int64_t)c.groups_k * kSplitGS * kSplitBK;
    const int64_t real = (int64_t)M * K, all = rows * kpad;
    // The last round: two workgroups that share a CU take 2000 cycles a slice, one alone 1700.
    // Where whole 128-row tiles lose half of their rate to it and to padding, a little over one
    // or two tiles per CU, the smaller fp32 tiles are faster (32 -> 432 3x3 stride 2, 284 tiles:
    // 1.30; 280 -> 1824@21x21 with a residual, 525: 1.26; 624 -> 448@46x46, 268: 1.09).
    const int64_t t128 = rows / 128 * ((ntot + 63) / 64) * d->group;
    if (c.bm == 128 && !c.sk && t128 > cus) {
        const int64_t rem = t128 % (2 * cus);
        const int64_t cycles = t128 / (2 * cus) * 2000 + (rem == 0 ? 0 : rem <= cus ? 1700 : 2000);
        if (1000. * t128 / ((double)cycles * cus) * real < 0.5 * all) return false;
    }
    if (split_pw2_shape(d)) return 20 * real >= 14 * all;
    const int least = d->kh * d->kw == 1 ? 15 : M > 64 ? 14 : 13; // twentieths
    if (20 * real < least * all || c.groups_k < 3 || (M > 64 && 5 * K < 4 * kpad)) return false;
    // Channel tails pay from one and a half 64-row tiles per CU (614 -> 376, 216 tiles: 1.30).
    if (d->c / d->group % 8 != 0 && 2 * tiles64 < 3 * cus) return false;
    // 64-row tiles, two to a CU, with 1-pixel loads: a little over one per CU, or two to three,
    // leave most of the last round empty, where smaller fp32 tiles do not (112 -> 192 3x3
    // stride 2, 273 tiles: 1.11; 176 -> 64, 601 tiles: 1.13); under one per CU the fp32 tiles
    // split a K of 1536 and more (464 -> 152 3x3 stride 2, 192 tiles: 75 -> 93).
    if (c.bm == 64 && tiles64 < cus && K >= 1536) return false;
    return c.bm == 128 || !((tiles64 > cus && 4 * tiles64 < 5 * cus) || (tiles64 > 2 * cus && tiles64 < 3 * cus));
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
