// split_core.h - fp32 matrix products on the bf16 matrix cores (gfx950).
//
// An fp32 value is the sum of three bf16 values: hi = bf16(v), mid = bf16(v - hi), lo the
// rest (8 significant bits each, both differences exact; from 2^-110 up the sum is exact,
// below that low bits can fall under bf16's least number, 2^-133, and the sum is off by
// less than that). A product a*b is then nine bf16 products, each exact in fp32; the six
// largest are accumulated here, in fp32, by v_mfma_f32_16x16x32_bf16. Of the three left
// out mid*lo and lo*mid are below 2^-25 of |a*b| each and lo*lo below 2^-34, so together
// they can reach the half unit, 2^-24, by which a lone product is rounded (one-term sums:
// largest error 1.65 x 2^-24, root mean square 0.435 x 2^-24 against 0.424 for fp32); sums
// of 64 terms and more are closer to 64 bits than on the fp32 MFMA (split_mfma). Six
// products at 16x the fp32 MFMA rate leave 2.67x its throughput (157 -> 419 TFLOP/s peak).
//
// Operands that the parts cannot carry give what fp32 arithmetic gives: a wave that meets
// them computes its accumulators again on the fp32 MFMA (fp32_product).
//  * Infinities, NaN and magnitudes that round to infinity turn every accumulator they
//    reach into an infinity or NaN.
//  * Weights that lose bits (times activations of any size), or of split_weight_limit and
//    more, are packed as NaN (conv_pack_split_kernel), which does the same.
//  * Activations that lose bits are off by less than 2^-133 times a weight under the limit:
//    over all of K by 2^-104 at most, 2^-24 of any accumulator of 2^-80 and more. Threads
//    note whether they split one; where they did, accumulators below 2^-80, zeros among
//    them, are computed again.
//  * Nonzero accumulators below 2^-104 are computed again in any case: six products round
//    at fp32's least number where fp32 rounds one.
//
// A operand (weights): split once when they are packed, laid out as the MFMA
// reads them, [K/8][3 planes][rows][8 k]: each wave loads its rows' fragments
// straight into registers, one 16-byte load per lane and plane.
// B operand (activations): each thread loads 8 consecutive k of one column,
// splits them (6 VALU operations per value) and stores three 16-byte runs to
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

// Two values to their three bf16 parts, packed (first value in the low half). The low 16 bits
// of `lost` take what the parts leave out: for values they carry, lo is exactly the upper
// half of what remains.
__device__ __forceinline__ void split2(float v0, float v1, uint32_t &hi, uint32_t &mid, uint32_t &lo, uint32_t &lost) {
    const bf16x2 h = __builtin_convertvector((f32x2){v0, v1}, bf16x2);
    hi = __builtin_bit_cast(uint32_t, h);
    const float r0 = v0 - __builtin_bit_cast(float, hi << 16);
    const float r1 = v1 - __builtin_bit_cast(float, hi & 0xffff0000u);
    const bf16x2 m = __builtin_convertvector((f32x2){r0, r1}, bf16x2);
    mid = __builtin_bit_cast(uint32_t, m);
    const uint32_t q0 = __builtin_bit_cast(uint32_t, r0 - __builtin_bit_cast(float, mid << 16));
    const uint32_t q1 = __builtin_bit_cast(uint32_t, r1 - __builtin_bit_cast(float, mid & 0xffff0000u));
    lo = __builtin_amdgcn_perm(q1, q0, 0x07060302u); // both upper halves
    // by hand: as C the ORs are gathered into trees whose leaves stay in registers
    asm("v_or3_b32 %0, %0, %1, %2" : "+v"(lost) : "v"(q0), "v"(q1));
}

__device__ __forceinline__ void split8(const float (&v)[8], u32x4 &hi, u32x4 &mid, u32x4 &lo, uint32_t &lost) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t h, m, l;
        split2(v[2 * i], v[2 * i + 1], h, m, l, lost);
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

// Magnitudes from which an accumulator outweighs the bits that activations lose (kSumLeast)
// and below which six products round visibly more often than one (kSumUnder).
constexpr float kSumLeast = 0x1p-80f, kSumUnder = 0x1p-104f;

// Largest power of two that K weights below it keep under 2^29 in sum.
inline float split_weight_limit(int K) {
    int bits = 0;
    while (((int64_t)1 << bits) < K) ++bits;
    return __builtin_ldexpf(1.f, 29 - bits);
}

// Whether the lane holds an accumulator that is infinite, NaN, zero or below 2^-80 (zero is
// also what outputs that do not exist hold).
template <int TM, int TN>
__device__ __forceinline__ bool sums_suspect(const f32x4 (&acc)[TM][TN]) {
    float least = __builtin_inff(); // a NaN is passed over
    float sum[2] = {0.f, 0.f};      // keeps an infinity or NaN, as one of the two or as inf - inf
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                least = fminf(least, fminf(fabsf(acc[i][j][r]), fabsf(acc[i][j][r + 1])));
                sum[0] += acc[i][j][r];
                sum[1] += acc[i][j][r + 1];
            }
    const float t = sum[0] + sum[1];
    return !(fabsf(t) < __builtin_inff()) | (least < kSumLeast);
}

// Whether it holds an infinity, NaN or nonzero below 2^-104.
template <int TM, int TN>
__device__ __forceinline__ bool sums_bad(const f32x4 (&acc)[TM][TN]) {
    bool bad = false;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float v = fabsf(acc[i][j][r]);
                bad = bad | !(v < __builtin_inff()) | ((v != 0.f) & (v < kSumUnder));
            }
    return bad;
}

// Accumulators of one wave again in fp32, over octets of k: load(o, a, b) gives the lane's
// operand values of octet o, a[s][i] for row block i and b[s][j] for column block j at
// k = 8 * o + 4 * s + lane / 16. The next octet's loads are in flight under this one's
// MFMAs.
template <int TM, int TN, class Load>
__device__ __forceinline__ void fp32_product(int o0, int o1, f32x4 (&acc)[TM][TN], Load &load) {
    float a[2][TM], b[2][TN], an[2][TM], bn[2][TN];
    if (o0 < o1) load(o0, a, b);
#pragma unroll 1
    for (int o = o0; o < o1; ++o) {
        load(o + 1, an, bn);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][i], b[s][j], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int i = 0; i < TM; ++i) a[s][i] = an[s][i];
#pragma unroll
            for (int j = 0; j < TN; ++j) b[s][j] = bn[s][j];
        }
    }
}

} // namespace spinn
