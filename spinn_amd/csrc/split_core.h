// split_core.h - fp32 matrix products on the bf16 matrix cores (gfx950).
//
// An fp32 value is exactly the sum of three bf16 values: hi = bf16(v),
// mid = bf16(v - hi), lo = bf16(v - hi - mid) (8 significant bits each, both
// differences exact). A product a*b is then nine bf16 products, each exact in
// fp32; the six largest are accumulated here, in fp32, by
// v_mfma_f32_16x16x32_bf16. The three left out (mid*lo, lo*mid, lo*lo) are below
// 2^-25 of |a*b|, under the rounding of the fp32 sums themselves. Six products at
// 16x the fp32 MFMA rate leave 2.67x its throughput (157 -> 419 TFLOP/s peak).
//
// Values that three bf16 parts cannot carry through a product turn every accumulator
// they reach into NaN or infinity (infinities, NaN, magnitudes that round to infinity)
// or leave it tiny (below 2^-110 the low parts fall under bf16's least number, 2^-133).
// A wave that finds such an accumulator after its K loop computes all of its own again
// on the fp32 MFMA (fp32_product), so these inputs give what fp32 arithmetic gives.
//
// A operand (weights): split once when they are packed, laid out as the MFMA
// reads them, [K/8][3 planes][rows][8 k]: each wave loads its rows' fragments
// straight into registers, one 16-byte load per lane and plane.
// B operand (activations): each thread loads 8 consecutive k of one column,
// splits them (5.5 VALU operations per value) and stores three 16-byte runs to
// LDS, [octet of k][3 planes][columns (+2)][8 k]; the MFMA reads them back as
// 16-byte fragments.
#pragma once
#include "mfma_core.h"

namespace spinn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kSplitBK = 32; // k per LDS slice: 4 octets, one MFMA step

constexpr int kSplitGS = 2;  // slices per LDS buffer (one barrier per group of slices)
constexpr int kSplitBN = 64; // columns of an output tile

// Output tile BM x 64 over 4 waves stacked along M, each TM x 4 blocks of 16x16
// (v_mfma_f32_16x16x32_bf16: operand lane l holds row or column l%16, k = 8*(l/16)..+7;
// accumulator element r of lane l is D[4*(l/16) + r][l%16]). Stacking along M loads each
// weight once per workgroup and splits each activation once per BM rows. CW: neighbouring
// columns per staging thread. Column c of the tile sits at LDS position
// (c % CW) * (64 / CW) + c / CW, so the threads' 16-byte stores are contiguous and a
// lane's accumulators hold CW neighbouring columns (CW-wide residual loads and stores).
template <int BM_, int CW_>
struct SplitTiling {
    static constexpr int BM = BM_, CW = CW_;
    static constexpr int WM = BM / 4, TM = WM / 16, TN = 4;
    static constexpr int NQ = TN / CW;
    // first of the CW neighbouring columns that blocks q, q + NQ, ... of a lane hold
    __device__ static __forceinline__ int col0(int q, int lane) { return (q * 16 + (lane & 15)) * CW; }
};

// Two values to their three bf16 parts, packed (first value in the low half).
__device__ __forceinline__ void split2(float v0, float v1, uint32_t &hi, uint32_t &mid, uint32_t &lo) {
    const bf16x2 h = __builtin_convertvector((f32x2){v0, v1}, bf16x2);
    hi = __builtin_bit_cast(uint32_t, h);
    const float r0 = v0 - __builtin_bit_cast(float, hi << 16);
    const float r1 = v1 - __builtin_bit_cast(float, hi & 0xffff0000u);
    const bf16x2 m = __builtin_convertvector((f32x2){r0, r1}, bf16x2);
    mid = __builtin_bit_cast(uint32_t, m);
    const float q0 = r0 - __builtin_bit_cast(float, mid << 16);
    const float q1 = r1 - __builtin_bit_cast(float, mid & 0xffff0000u);
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){q0, q1}, bf16x2));
}

__device__ __forceinline__ void split8(const float (&v)[8], u32x4 &hi, u32x4 &mid, u32x4 &lo) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t h, m, l;
        split2(v[2 * i], v[2 * i + 1], h, m, l);
        hi[i] = h;
        mid[i] = m;
        lo[i] = l;
    }
}

// LDS buffer of one group of slices of the split B operand: [octet][plane][64 + 2] runs
// of 16 bytes.
constexpr int kSplitRow = kSplitBN + 2;
constexpr int kSplitRuns = kSplitGS * 4 * 3 * kSplitRow;
__device__ __forceinline__ int split_at(int plane, int oct, int pos) { return (oct * 3 + plane) * kSplitRow + pos; }

// Packed split weights of one group: [octet][plane][rows_p][8 bf16]; rows_p is the
// row count padded to kSplitRowPad, octets padded to whole slices, padding zero.
constexpr int kSplitRowPad = 64;
struct SplitPlanes {
    const float *base;
    uint32_t bytes;
    int rows_p;
    int octs; // multiple of 4
};

// A operand fetcher: one slice of the wave's TM row blocks, straight to registers.
// Rows past rows_p (tiles wider than the padding) repeat the last row; their
// results are never stored.
template <int TM>
struct PlanesA {
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t voff[TM];
    uint32_t plane_bytes, slice_bytes;
    int last;
    __device__ __forceinline__ void init(const SplitPlanes &p, int row0, int lane) {
        rsrc = make_rsrc(p.base, p.bytes);
        plane_bytes = (uint32_t)p.rows_p * 16u;
        slice_bytes = plane_bytes * 12u;
        last = p.octs / 4 - 1;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int row = min(row0 + i * 16 + (lane & 15), p.rows_p - 1);
            voff[i] = (uint32_t)(lane >> 4) * 3u * plane_bytes + (uint32_t)row * 16u;
        }
    }
    // Slices past the last repeat it (their values are never used).
    __device__ __forceinline__ void fetch(int slice, bf16x8 (&a)[TM][3]) const {
        const uint32_t s = (uint32_t)min(slice, last) * slice_bytes;
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int i = 0; i < TM; ++i)
                a[i][p] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
                                                         rsrc, (int)voff[i], (int)(s + p * plane_bytes), 0));
    }
};

template <int T>
__device__ __forceinline__ void read_frags(const u32x4 *lds, int slice, int pos0, int lane, bf16x8 (&f)[T][3]) {
    const u32x4 *q = lds + split_at(0, lane >> 4, pos0 + (lane & 15));
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int j = 0; j < T; ++j) f[j][p] = __builtin_bit_cast(bf16x8, q[split_at(p, slice * 4, j * 16)]);
}

// Product Q of the six of one slice, over column blocks J0..J0+NJ. hi*hi (Q = 0) goes to
// `acc`, the five small ones to `low`, added to it once after the K loop: the running
// sum is then rounded once per 32 k, not at every product (1x1, K = 1024: 4.6e-7 ->
// 1.4e-7 against 64 bits). Consecutive MFMAs go to different accumulators.
template <int Q, int TM, int TN, int J0, int NJ>
__device__ __forceinline__ void split_mfma(const bf16x8 (&a)[TM][3], const bf16x8 (&b)[NJ][3],
                                           f32x4 (&acc)[TM][TN], f32x4 (&low)[TM][TN]) {
    constexpr int pa[6] = {0, 0, 1, 1, 0, 2};
    constexpr int pb[6] = {0, 1, 0, 1, 2, 0};
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            f32x4 &c = Q == 0 ? acc[i][J0 + j] : low[i][J0 + j];
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][pa[Q]], b[j][pb[Q]], c, 0, 0, 0);
        }
}

// True when any accumulator of the wave is infinite, NaN, or nonzero below 2^-80, which
// sums of ordinary values do not cancel down to (their residue is 2^-24 of a term).
template <int TM, int TN>
__device__ __forceinline__ bool out_of_range(const f32x4 (&acc)[TM][TN]) {
    constexpr uint32_t kTiny = (127u - 80u) << 23;
    float s = 0.f;         // v * 0 is 0 for finite v and NaN otherwise; a NaN survives the sums
    uint32_t low = ~0u;    // least |v| - 1 as bits: zero wraps to the largest
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                s += acc[i][j][r] * 0.f;
                low = min(low, (__builtin_bit_cast(uint32_t, acc[i][j][r]) & 0x7fffffffu) - 1u);
            }
    return __any(s != s || low < kTiny);
}

// Accumulators of one wave again in fp32: av(i, k) and bv(j, k) give the lane's
// operand values for row block i and column block j.
template <int TM, int TN, class AV, class BV>
__device__ __forceinline__ void fp32_product(int k0, int k1, int lane, f32x4 (&acc)[TM][TN], const AV &av,
                                             const BV &bv) {
#pragma unroll 1
    for (int k = k0; k < k1; k += 4) {
        const int kk = k + (lane >> 4);
        float a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = av(i, kk);
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = bv(j, kk);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
}

} // namespace spinn
