// orb_kernels.hip -- gfx950 kernels of the ORB front end.
//
// Pipeline per image (one launch per stage covers every job of a run):
//   pyramid_kernel levels 1 .. from level 0 (8-bit fixed point bilinear,
//                  ORBextractor.cc:1677), several levels per launch
//   level_kernel   every level's 7x7 sigma-2 blur (ORBextractor.cc:1607-1615)
//                  and FAST-9 with per-cell non-max suppression at both
//                  thresholds (ORBextractor.cc:1075-1142), from one LDS tile
//   octree_kernel  the per-cell iniThFAST/minThFAST retry, then
//                  DistributeOctTree as a per-level workgroup quadtree
//                  (ORBextractor.cc:688-1033)
//   describe_kernel IC_Angle + rotated BRIEF + output assembly
//                  (ORBextractor.cc:94-204, 1590-1648)
// plus stereo matching (Frame.cc:831-1082) and brute-force Hamming matching.
//
// All float code is compiled with -ffp-contract=off: every float statement
// that the reference evaluates is evaluated here with the same operations in
// the same order, so results are bit-identical to the CPU statement.
#include <hip/hip_runtime.h>
#include <float.h>
#include <limits.h>

#include "orb_types.h"

__constant__ __align__(16) signed char c_pattern[1024] = {   // BRIEF pairs, x0,y0,x1,y1
#include "orb_pattern.inc"
};
__constant__ __align__(16) uint4 c_icmask[4 * 16 * 3];   // orientation disc byte masks [alignment][|v|][16 bytes]
// 7x7 sigma-2 blur as two matrix products: the band matrices of the integer
// taps (8 bytes of k a lane; the second one's k as level_kernel's first product
// leaves its rows) and the sums that undo the signed operands' offsets.
__constant__ __align__(16) uint2 c_band[2][64];
__constant__ int c_bandsum[2];

// umax16: the orientation disc half-widths of the constructor
// (ORBextractor.cc:542-570).  Byte k of dword c of a patch row whose first
// dword starts `al` pixels left of u = -15 holds u = 4c + k - 15 - al; its
// mask byte is 0xFF iff |u| <= umax[|v|].
extern "C" hipError_t orb_upload_constants(const int* umax16, const int* gauss7)
{
    unsigned m[4 * 16 * 12];
    for (int al = 0; al < 4; al++)
        for (int av = 0; av < 16; av++)
            for (int c = 0; c < 12; c++) {
                unsigned w = 0;
                for (int k = 0; k < 4; k++) {
                    const int u = 4 * c + k - 15 - al;
                    if ((u < 0 ? -u : u) <= umax16[av]) w |= 0xFFu << (8 * k);
                }
                m[(al * 16 + av) * 12 + c] = w;
            }
    hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_icmask), m, sizeof(m));
    if (e != hipSuccess) return e;
    uint2 band[2][64];
    int sum = 0;
    for (int i = 0; i < 7; i++) sum += gauss7[i];
    if (sum > 257) return hipErrorInvalidValue;         // a row sum must fit 16 bits
    for (int lane = 0; lane < 64; lane++) {
        const int n = lane & 15, g = lane >> 4;
        unsigned w[2][2] = {};
        for (int j = 0; j < 8; j++) {
            // columns: byte k of the window that starts 4 pixels left of the
            // tile's 16; rows: 4 of each of two 16-row products
            const int tap[2] = {8 * g + j - n - 1, (j < 4 ? 4 * g + j : 12 + 4 * g + j) - n};
            for (int d = 0; d < 2; d++)
                if (tap[d] >= 0 && tap[d] < 7) w[d][j >> 2] |= (unsigned)gauss7[tap[d]] << (8 * (j & 3));
        }
        for (int d = 0; d < 2; d++) band[d][lane] = make_uint2(w[d][0], w[d][1]);
    }
    e = hipMemcpyToSymbol(HIP_SYMBOL(c_band), band, sizeof(band));
    if (e != hipSuccess) return e;
    const int bias[2] = {128 * sum - 32768, sum * (32768 + 128)};
    return hipMemcpyToSymbol(HIP_SYMBOL(c_bandsum), bias, sizeof(bias));
}

// ------------------------------------------------------------------ helpers
// Loads of 16, 8 and 4 bytes at 4-byte aligned global addresses, marked as
// global so that they are issued as global (not flat) loads.
typedef unsigned orb_v4u __attribute__((ext_vector_type(4), aligned(4)));
typedef unsigned orb_v2u __attribute__((ext_vector_type(2), aligned(4)));
__device__ __forceinline__ uint4 gload16(const uint8_t* p)
{
    const orb_v4u v = *(const __attribute__((address_space(1))) orb_v4u*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint2 gload8(const uint8_t* p)
{
    const orb_v2u v = *(const __attribute__((address_space(1))) orb_v2u*)p;
    return make_uint2(v.x, v.y);
}
// 8 bytes that no thread writes during the kernel, at a wave-uniform address:
// constant address space, so that it is a scalar load.
__device__ __forceinline__ uint2 cload8(const void* p)
{
    const orb_v2u v = *(const __attribute__((address_space(4))) orb_v2u*)p;
    return make_uint2(v.x, v.y);
}
typedef unsigned orb_u32a1 __attribute__((aligned(1)));
__device__ __forceinline__ unsigned gload4u(const uint8_t* p)   // any alignment
{
    return *(const __attribute__((address_space(1))) orb_u32a1*)p;
}
// Stores through global (not flat) addresses.
__device__ __forceinline__ void gstore4(uint8_t* p, unsigned v) { *(__attribute__((address_space(1))) unsigned*)p = v; }
__device__ __forceinline__ void gstore1(uint8_t* p, uint8_t v) { *(__attribute__((address_space(1))) uint8_t*)p = v; }
__device__ __forceinline__ void gstore8(unsigned long long* p, unsigned long long v)
{
    *(__attribute__((address_space(1))) unsigned long long*)p = v;
}
__device__ __forceinline__ unsigned long long gload8u64(const unsigned long long* p)
{
    return *(const __attribute__((address_space(1))) unsigned long long*)p;
}
__device__ __forceinline__ uint8_t gload1(const uint8_t* p) { return *(const __attribute__((address_space(1))) uint8_t*)p; }
__device__ __forceinline__ void gstore2(uint8_t* p, unsigned short v)
{
    *(__attribute__((address_space(1))) unsigned short*)p = v;
}
__device__ __forceinline__ void gstore16(uint8_t* p, uint4 v)
{
    *(__attribute__((address_space(1))) orb_v4u*)p = orb_v4u{v.x, v.y, v.z, v.w};
}
__device__ __forceinline__ unsigned gload4(const uint8_t* p)
{
    return *(const __attribute__((address_space(1))) unsigned*)p;
}

__device__ __forceinline__ int reflect101(int i, int n)
{
    if (i < 0) i = -i;
    if (i >= n) i = 2 * n - 2 - i;
    return i < 0 ? 0 : (i >= n ? n - 1 : i);
}

__device__ __forceinline__ int find_segment(const int* starts, int n, int x)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (starts[mid] <= x) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Sum over the 16 lanes of a DPP row (all of them active); every lane of the
// row receives the total.
__device__ __forceinline__ unsigned row16_sum(unsigned v)
{
    v += (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false);    // quad_perm [1,0,3,2]
    v += (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false);    // quad_perm [2,3,0,1]
    v += (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, false);   // row_half_mirror
    v += (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x140, 0xF, 0xF, false);   // row_mirror
    return v;
}

// The dispatcher sends workgroup b to XCD b % 8, and each XCD has its own
// L2.  This bijection on [0, n) hands XCD x the contiguous logical range
// [x*q + min(x, r), ...) (q = n / 8, r = n % 8), so neighbouring tiles, whose
// halos share cache lines, and the keypoints of one image meet in one L2.
#define ORB_NUM_XCD 8
__device__ __forceinline__ int xcd_block(int b, int n)
{
    const unsigned q = (unsigned)n / ORB_NUM_XCD, r = (unsigned)n % ORB_NUM_XCD;
    const unsigned x = (unsigned)b % ORB_NUM_XCD, i = (unsigned)b / ORB_NUM_XCD;
    return (int)(x * q + min(x, r) + i);
}

__device__ __forceinline__ int lanes_below(unsigned long long mask)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
}

// ================================================================ level
// One workgroup per 64x32 (or 64x16) output tile of pyramid level l, the tiles
// of all levels in one launch:
//   1. level pixels for the tile plus a 4-px halo (REFLECT_101 at the level
//      edges) into LDS;
//   2. its 7x7 sigma-2 blur (ORBextractor.cc:1607-1615);
//   3. FAST-9 arc strength for the tile plus a 1-px ring, computed exactly only
//      for pixels that pass a necessary cardinal-point test, after compaction;
//   4. per-cell non-max suppression at iniThFAST and at minThFAST: a neighbour
//      counts only if it lies in the same 30-px cell's detection area, which is
//      exactly cv::FAST run on that cell's window (ORBextractor.cc:1075-1142);
//   5. candidates of either threshold appended to the level's key list (one
//      entry says which), and a per-cell flag set when the cell has an iniThFAST survivor.  The quadtree
//      kernel keeps minThFAST candidates only for cells without that flag,
//      which is the reference's per-cell retry.
#define LT_W ORB_TILE_W
#define LT_HALO 4
#define LP_W (LT_W + 2 * LT_HALO)      // 72 bytes = 18 dwords
#define LP_WD (LP_W / 4)
#define LK_CAP 1536                  // per-tile candidates, both thresholds

typedef unsigned short orb_us2 __attribute__((ext_vector_type(2)));
typedef int orb_v4i __attribute__((ext_vector_type(4)));

// The largest t + 1 at which the pixel is a FAST-9 corner: the largest minimum
// over the 16 runs of 9 contiguous ring pixels less the centre, or the centre
// less the smallest maximum.  The runs starting at k and k + 1 share 8 pixels:
// the larger of their minima is min(minimum of the 8, max of the two outer
// ones), so 8 runs of 8 serve all 16.  Register j holds the opposite pixels j
// and j + 8 of the ring (Bresenham radius 3, in OpenCV's makeOffsets(16)
// order), so that a step along the ring is the next register and one past the
// end the halves exchanged, which the packed instructions select by themselves:
// 23 of them a side, where the 16 runs one by one took 44 and 16 to prepare.
// level_kernel on 128 images of 1241 x 376 558 -> 500 us, on 64 of four sizes
// 311 -> 280.
__device__ __forceinline__ int fast_strength(const uint8_t* p, int stride)
{
    const unsigned v = p[0];
    const unsigned r[16] = {p[3 * stride],      p[3 * stride + 1],  p[2 * stride + 2],  p[stride + 3],
                            p[3],               p[-stride + 3],     p[-2 * stride + 2], p[-3 * stride + 1],
                            p[-3 * stride],     p[-3 * stride - 1], p[-2 * stride - 2], p[-stride - 3],
                            p[-3],              p[stride - 3],      p[2 * stride - 2],  p[3 * stride - 1]};
    orb_us2 R[9];
#pragma unroll
    for (int j = 0; j < 8; j++) R[j] = __builtin_bit_cast(orb_us2, r[j] | (r[j + 8] << 16));
    auto turn = [](orb_us2 x) { return __builtin_shufflevector(x, x, 1, 0); };
    R[8] = turn(R[0]);
    // for each odd s = 2 i + 1: pairs, fours and eights from s on, and the two outer pixels
    orb_us2 N2[4], X2[4], N4[4], X4[4], B[4], K[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        N2[i] = __builtin_elementwise_min(R[2 * i + 1], R[2 * i + 2]);
        X2[i] = __builtin_elementwise_max(R[2 * i + 1], R[2 * i + 2]);
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        N4[i] = __builtin_elementwise_min(N2[i], i < 3 ? N2[(i + 1) & 3] : turn(N2[0]));
        X4[i] = __builtin_elementwise_max(X2[i], i < 3 ? X2[(i + 1) & 3] : turn(X2[0]));
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const orb_us2 n8 = __builtin_elementwise_min(N4[i], i < 2 ? N4[(i + 2) & 3] : turn(N4[i - 2]));
        const orb_us2 x8 = __builtin_elementwise_max(X4[i], i < 2 ? X4[(i + 2) & 3] : turn(X4[i - 2]));
        const orb_us2 o = turn(R[2 * i + 1]);
        B[i] = __builtin_elementwise_min(n8, __builtin_elementwise_max(R[2 * i], o));
        K[i] = __builtin_elementwise_max(x8, __builtin_elementwise_min(R[2 * i], o));
    }
    const orb_us2 b = __builtin_elementwise_max(__builtin_elementwise_max(B[0], B[1]), __builtin_elementwise_max(B[2], B[3]));
    const orb_us2 k = __builtin_elementwise_min(__builtin_elementwise_min(K[0], K[1]), __builtin_elementwise_min(K[2], K[3]));
    // A pixel is a FAST-9 corner at threshold t iff strength > t, and then
    // OpenCV's cornerScore equals strength - 1.
    const int bright = (int)max((unsigned)b.x, (unsigned)b.y) - (int)v, dark = (int)v - (int)min((unsigned)k.x, (unsigned)k.y);
    return max(max(bright, dark), 0);
}

// Necessary condition for strength > t, on two pixels at once (16-bit
// lanes): a 9-run covers two circularly adjacent cardinal points (ring
// positions 0, 4, 8, 12), all brighter than v+t or all darker than v-t.
__device__ __forceinline__ unsigned fast_maybe2(unsigned v, unsigned p0, unsigned p4, unsigned p8, unsigned p12,
                                                unsigned t2)
{
    const orb_us2 V = __builtin_bit_cast(orb_us2, v), T = __builtin_bit_cast(orb_us2, t2);
    const orb_us2 hi = V + T;                                   // <= 510, no wrap
    const orb_us2 lo = __builtin_elementwise_sub_sat(V, T);     // max(v - t, 0)
    const orb_us2 a = __builtin_bit_cast(orb_us2, p0), b = __builtin_bit_cast(orb_us2, p4);
    const orb_us2 c = __builtin_bit_cast(orb_us2, p8), d = __builtin_bit_cast(orb_us2, p12);
    // Some circularly adjacent pair (0,4), (4,8), (8,12), (12,0) is brighter
    // than hi <=> (0 or 8) and (4 or 12) are <=> min(max(p0, p8),
    // max(p4, p12)) > hi: opposite points never pair up.  Darker likewise
    // with max(min, min) < lo.  Nonzero lane <=> the pixel may pass.
    const orb_us2 M = __builtin_elementwise_min(__builtin_elementwise_max(a, c), __builtin_elementwise_max(b, d));
    const orb_us2 m = __builtin_elementwise_max(__builtin_elementwise_min(a, c), __builtin_elementwise_min(b, d));
    const orb_us2 r = __builtin_elementwise_max(__builtin_elementwise_sub_sat(M, hi), __builtin_elementwise_sub_sat(lo, m));
    return __builtin_bit_cast(unsigned, r);
}

// Bytes 0 and 2 (lo_bytes) or 1 and 3 (hi_bytes) of a dword, zero-extended
// into the two 16-bit lanes.
__device__ __forceinline__ unsigned lo_bytes(unsigned x) { return __builtin_amdgcn_perm(0u, x, 0x0C020C00u); }
__device__ __forceinline__ unsigned hi_bytes(unsigned x) { return __builtin_amdgcn_perm(0u, x, 0x0C030C01u); }

// Four adjacent pixels of cv::resize INTER_LINEAR 8U from the source rows at
// byte offsets o0, o1 of base (the LDS window, or the level in global memory
// with 32-bit offsets): horizontal 11-bit taps (a0 | a1 << 16) per column,
// vertical taps yb = b0 | b1 << 16, rounding shift by 22.
// - All terms are non-negative, so the shift is done unsigned.  (A signed
//   shift with a [0, 255] clamp of lanes 0 and 1 is lowered by the gfx950
//   backend to v_ashr_pk_u8_i32, whose upper result half then leaked into
//   bytes 2 and 3.)
// - Every factor is below 2^24 (taps <= 2048, S <= 255 * 4096), so the
//   products are 24-bit multiplies (v_mul_u32_u24, full rate) rather than
//   32-bit ones (v_mul_lo_u32, quarter rate).
typedef unsigned short orb_u16x2 __attribute__((ext_vector_type(2)));

// The vertical pass on the horizontal sums S0, S1 (each <= 255 * 2049) with
// the row taps b0, b1, rounded as OpenCV's generic scalar code does
// ((S0*b0 + S1*b1 + 2^21) >> 22) or as its SSE2 kernel VResizeLinearVec_32s8u
// does (S >> 4 as int16, _mm_mulhi_epi16 by the taps, + 2, >> 2).  Neither
// needs a clamp or a saturation: every tap pair sums to 2047..2049 (two
// roundings of values summing to 2048), so the scalar form is at most
// (255 * 2049 * 2049 + 2^21) >> 22 = 255, the SSE2 one at most
// (2 * ((32655 * 2049) >> 17) + 2) >> 2 = 255, and S >> 4 <= 32655 fits int16.
// MODE 0: scalar, 1: SSE2, 2: SSE2 where sse != 0.
template <int MODE>
__device__ __forceinline__ unsigned vresize(unsigned S0, unsigned S1, unsigned b0, unsigned b1, unsigned sse)
{
    const unsigned vc = (__umul24(S0, b0) + __umul24(S1, b1) + (1u << 21)) >> 22;
    const unsigned vs = ((__umul24(S0 >> 4, b0) >> 16) + (__umul24(S1 >> 4, b1) >> 16) + 2u) >> 2;
    return MODE == 0 ? vc : (MODE == 1 ? vs : (sse ? vs : vc));
}

// High 32 bits of a 24 x 24-bit product (v_mul_hi_u32_u24, full rate): the
// operands are masked to 24 bits, which is what lets the compiler pick it.
__device__ __forceinline__ unsigned mulhi_u24(unsigned a, unsigned b)
{
    return (unsigned)(((unsigned long long)(a & 0xFFFFFFu) * (unsigned long long)(b & 0xFFFFFFu)) >> 32);
}

template <int M>
struct ModeTag {
    static constexpr int value = M;
};

template <typename BytePtr>
__device__ __forceinline__ unsigned resize4(BytePtr base, unsigned o0, unsigned o1, const int* sxk, const int* nxk,
                                            const int* tap, int yb, const unsigned* sse)
{
    const unsigned b0 = (unsigned)yb & 0xFFFFu, b1 = (unsigned)yb >> 16;
    unsigned d = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const unsigned a0 = (unsigned)tap[k] & 0xFFFFu, a1 = (unsigned)tap[k] >> 16;
        const unsigned S0 = __umul24(base[o0 + sxk[k]], a0) + __umul24(base[o0 + nxk[k]], a1);
        const unsigned S1 = __umul24(base[o1 + sxk[k]], a0) + __umul24(base[o1 + nxk[k]], a1);
        d |= vresize<2>(S0, S1, b0, b1, sse[k]) << (8 * k);
    }
    return d;
}

// Four output pixels from the source rows at q0, q1 (dword pointers to the
// dword that holds byte b0 of the four pixels' span, shb = b0 & 3): a source
// row is three aligned dword reads realigned by two v_alignbyte, each pixel's
// tap pair (p[sx], p[nx]) one v_perm into 16-bit lanes (sel), and S one
// v_dot2_u32_u16 with the packed taps (a0 | a1 << 16).
template <int MODE>
__device__ __forceinline__ unsigned resize_dword(const unsigned* q0, const unsigned* q1, unsigned shb, const unsigned* sel,
                                                 const int* tap, unsigned ybv, const unsigned* sse)
{
    const unsigned w00 = __builtin_amdgcn_alignbyte(q0[1], q0[0], shb);
    const unsigned w01 = __builtin_amdgcn_alignbyte(q0[2], q0[1], shb);
    const unsigned w10 = __builtin_amdgcn_alignbyte(q1[1], q1[0], shb);
    const unsigned w11 = __builtin_amdgcn_alignbyte(q1[2], q1[1], shb);
    if constexpr (MODE == 1) {
        // SSE2 rounding with the horizontal taps scaled by 16: S16 = 16 S, so
        // S16 & 0xFFFF00 = (S >> 4) << 8 (S16 < 2^23), and the high word of
        // its product with b << 8 is ((S >> 4) * b) >> 16 in one
        // v_mul_hi_u32_u24.  t = h0 + h1 + 2 <= 1023 fits a 16-bit lane: the
        // >> 2 is done two pixels at a time and the four bytes gathered by
        // one v_perm.
        const unsigned bs0 = (ybv << 8) & 0xFFFF00u, bs1 = (ybv >> 8) & 0xFFFF00u;
        unsigned t[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const orb_u16x2 tk = __builtin_bit_cast(orb_u16x2, (unsigned)tap[k] << 4);
            const unsigned S0 = __builtin_amdgcn_udot2(
                __builtin_bit_cast(orb_u16x2, __builtin_amdgcn_perm(w01, w00, sel[k])), tk, 0u, false);
            const unsigned S1 = __builtin_amdgcn_udot2(
                __builtin_bit_cast(orb_u16x2, __builtin_amdgcn_perm(w11, w10, sel[k])), tk, 0u, false);
            t[k] = mulhi_u24(S0 & 0xFFFF00u, bs0) + mulhi_u24(S1 & 0xFFFF00u, bs1) + 2u;
        }
        const orb_u16x2 two = {2, 2};
        const unsigned u01 = __builtin_bit_cast(unsigned, __builtin_bit_cast(orb_u16x2, t[0] | (t[1] << 16)) >> two);
        const unsigned u23 = __builtin_bit_cast(unsigned, __builtin_bit_cast(orb_u16x2, t[2] | (t[3] << 16)) >> two);
        return __builtin_amdgcn_perm(u23, u01, 0x06040200u);
    } else {
        const unsigned bv0 = ybv & 0xFFFFu, bv1 = ybv >> 16;
        unsigned d = 0;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const orb_u16x2 tk = __builtin_bit_cast(orb_u16x2, (unsigned)tap[k]);
            const unsigned S0 = __builtin_amdgcn_udot2(
                __builtin_bit_cast(orb_u16x2, __builtin_amdgcn_perm(w01, w00, sel[k])), tk, 0u, false);
            const unsigned S1 = __builtin_amdgcn_udot2(
                __builtin_bit_cast(orb_u16x2, __builtin_amdgcn_perm(w11, w10, sel[k])), tk, 0u, false);
            d |= vresize<MODE>(S0, S1, bv0, bv1, sse[k]) << (8 * k);
        }
        return d;
    }
}

// ============================================================== pyramid
// cv::resize INTER_LINEAR 8U of levels base + 1 .. base + m, each from the
// level before (ComputePyramid, ORBextractor.cc:1677).  A workgroup takes one
// tile of the last level and computes, level by level in LDS, what that tile
// needs of each; the levels' tiles overlap by a few pixels, and each pixel is
// written by the one workgroup that owns it (windows and ownership come from
// the host, by tile column and row).  At scale factor 1.2 all seven levels
// are one launch, with 1.4 times the pixels computed.  Bound: latency (one
// LDS round trip and barrier per level) in a single call, VALU in a batch.
// One image of 640 x 480 14.9 us, and every level's tiles after it 12.2 (9 with
// the tiles' later changes), where a launch per level that resized its own tile
// took 82; 128 images of 1241 x 376 148 + 566 us (725; 420 for the 566 now).
// The source index and 11-bit taps of each column and row come from the
// level's tables (computed on the host with OpenCV's double/float
// statements).
__device__ __forceinline__ void zero_job(const ImageJob& J)
{
    if (threadIdx.x < ORB_CNT_SLOTS) gstore4((uint8_t*)(J.counters + threadIdx.x), 0u);
    for (int i = threadIdx.x; i < J.nlevels * ORB_SEGS; i += blockDim.x)
        gstore4((uint8_t*)(J.lv[i / ORB_SEGS].segs + i % ORB_SEGS * ORB_SEG_STRIDE), 0u);
    // 32 threads per level, the levels side by side
    for (int l = threadIdx.x >> 5; l < J.nlevels; l += blockDim.x >> 5) {
        uint8_t* f = J.lv[l].cellflag;
        const int n = J.lv[l].ncells;
        for (int i = threadIdx.x & 31; i < n; i += 32) gstore1(f + i, 0);
    }
}

template <int V>
__global__ __launch_bounds__(ORB_CH_T) void pyramid_kernel(const ImageJob* __restrict__ jobs,
                                                             const RunTable* __restrict__ rt, int chain, int zero)
{
    constexpr int T = ORB_CH_T;
    __shared__ unsigned buf[2][ORB_CH_DWORDS + 4];
    __shared__ int2 s_row[2][ORB_CH_ROWS];
    const int tid = threadIdx.x;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int tpj = rt->chain_per_job[chain];
    const int job = tpj > 0 ? blk / tpj : find_segment(rt->chain_start[chain], rt->njobs, blk);
    const int t = blk - rt->chain_start[chain][job];
    const ImageJob& J = jobs[job];
    const ChainJob& C = J.ch[V][chain];
    const int m = C.m, base = C.base;
    const ChainWin* xr = C.xr + (size_t)(t % C.tiles_x) * (m + 1);
    const ChainWin* yr = C.yr + (size_t)(t / C.tiles_x) * (m + 1);
    if (zero && t == 0) zero_job(J);

    if (!C.staged) {
        // a window too large for LDS (m = 1): taps read from memory
        const LevelJob& L = J.lv[base + 1];
        const LevelJob& P = J.lv[base];
        const ChainWin cx = xr[1], cy = yr[1];
        const int nd = ((cx.o1 - 1) >> 2) - (cx.o0 >> 2) + 1;
        for (int e = tid; e < nd * (cy.o1 - cy.o0); e += T) {
            const int y = cy.o0 + e / nd, x = cx.o0 + 4 * (e % nd);
            int sxk[4], nxk[4], tap[4];
            unsigned sse[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint2 v = gload8((const uint8_t*)(L.xtab + min(x + k, L.w - 1)));
                sxk[k] = (int)v.x & 0x3FFFFFFF;
                nxk[k] = min(sxk[k] + 1, P.w - 1);
                sse[k] = v.x >> 30;
                tap[k] = (int)v.y;
            }
            const uint2 r = gload8((const uint8_t*)(L.ytab + y));
            gstore4(L.lvl + (unsigned)(y * L.pitch + x),
                    resize4((const __attribute__((address_space(1))) uint8_t*)P.lvl, __umul24(r.x & 0xFFFFu, P.pitch),
                            __umul24(r.x >> 16, P.pitch), sxk, nxk, tap, (int)r.y, sse));
        }
        return;
    }

    // Of level base + k: this thread's 4-column group's taps (thread tid
    // takes group tid % nd, rows tid / nd, + T / nd, ...), and one row entry.
    uint2 xt[4], yt;
    auto load_taps = [&](int k) {
        const LevelJob& L = J.lv[base + k];
        const int nd = xr[k].nd, c = tid - (int)(__umul24((unsigned)tid, xr[k].rcp) >> 20) * nd, x = xr[k].a + 4 * c;
#pragma unroll
        for (int q = 0; q < 4; q++) xt[q] = gload8((const uint8_t*)(L.xtab + min(x + q, L.w - 1)));
        yt = gload8((const uint8_t*)(L.ytab + min(yr[k].a + min(tid, ORB_CH_ROWS - 1), L.h - 1)));
    };
    {
        // the base window, in whole aligned dwords (level rows start 64-byte
        // aligned, so no read leaves its row's pitch); the input when it is not
        // level 0 itself
        const uint8_t* src = base == 0 ? J.src : J.lv[base].lvl;
        const int sp = base == 0 ? J.src_pitch : J.lv[base].pitch;
        const int nd = xr[0].nd, n = nd * (yr[0].b - yr[0].a + 1);
        const unsigned rcp = xr[0].rcp;            // e / nd, exact for e * nd < 2^20
        const uint8_t* s0 = src + (size_t)yr[0].a * sp + xr[0].a;
        load_taps(1);
        constexpr int Q = 6;
        for (int e0 = tid; e0 < n; e0 += Q * T) {
            unsigned d[Q];
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const int e = min(e0 + T * q, n - 1);
                const int r = (int)(__umul24((unsigned)e, rcp) >> 20);
                const unsigned off = (unsigned)(r * sp + 4 * (e - r * nd));
                d[q] = (sp & 3) == 0 ? gload4(s0 + off) : gload4u(s0 + off);
            }
#pragma unroll
            for (int q = 0; q < Q; q++)
                if (e0 + T * q < n) buf[0][e0 + T * q] = d[q];
        }
        if (tid < ORB_CH_ROWS) s_row[1][tid] = make_int2((int)yt.x, (int)yt.y);
    }
    __syncthreads();
#pragma unroll 1
    for (int k = 1; k <= m; k++) {
        const LevelJob& L = J.lv[base + k];
        const int sw = J.lv[base + k - 1].w;
        const ChainWin cx = xr[k], cy = yr[k];
        const int nd = cx.nd, nrows = cy.b - cy.a + 1;
        const int wx0 = xr[k - 1].a, wy0 = yr[k - 1].a, ws = xr[k - 1].nd;
        const int r0 = (int)(__umul24((unsigned)tid, cx.rcp) >> 20), rstep = (int)(((unsigned)T * cx.rcp) >> 20);
        const int c = tid - r0 * nd;
        const unsigned* src = buf[(k - 1) & 1];
        unsigned* dst = buf[k & 1];
        int sxk[4], nxk[4], tap[4];
        unsigned sse[4];                           // SSE2 rounding for the column (xtab bit 30)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int sx = (int)xt[q].x & 0x3FFFFFFF;
            sse[q] = xt[q].x >> 30;
            sxk[q] = sx - wx0;
            nxk[q] = min(sx + 1, sw - 1) - wx0;
            tap[q] = (int)xt[q].y;
        }
        if (k < m) load_taps(k + 1);               // in flight under this level's rows
        // Rounding of the window's columns: all scalar, all SSE2, or per
        // column where it reaches the last columns the SSE2 kernel leaves to
        // the scalar pass.
        const int rmode = L.rs_end == 0 ? 0 : (cx.b < L.rs_end ? 1 : 2);
        const int x = cx.a + 4 * c;
        const bool xin = x >= cx.o0 && x < cx.o1;
        const int pitch = L.pitch;
        uint8_t* out = L.lvl + (unsigned)(cy.a * pitch + x);
        auto emit = [&](int ey, unsigned d) {
            if (k < m) dst[ey * nd + c] = d;
            if (xin && cy.a + ey >= cy.o0 && cy.a + ey < cy.o1) gstore4(out + (unsigned)(ey * pitch), d);
        };
        if (r0 < rstep) {
            // The four pixels' source bytes usually lie within 8 bytes (scale
            // factors up to ~2.3).
            if (nxk[3] - sxk[0] <= 7) {
                const unsigned* wd = src + (sxk[0] >> 2);
                const unsigned shb = (unsigned)(sxk[0] & 3);
                unsigned sel[4];
#pragma unroll
                for (int q = 0; q < 4; q++)
                    sel[q] = 0x0C000C00u | ((unsigned)(nxk[q] - sxk[0]) << 16) | (unsigned)(sxk[q] - sxk[0]);
                auto rows = [&](auto mode) {
                    // two rows at a time, so that their LDS reads overlap
                    // (the second repeats the first where there is none)
                    for (int ey = r0; ey < nrows; ey += 2 * rstep) {
                        const int ez = ey + rstep < nrows ? ey + rstep : ey;
                        const int2 yv = s_row[k & 1][ey], zv = s_row[k & 1][ez];
                        const unsigned d = resize_dword<decltype(mode)::value>(
                            wd + __umul24(((unsigned)yv.x & 0xFFFFu) - wy0, ws),
                            wd + __umul24(((unsigned)yv.x >> 16) - wy0, ws), shb, sel, tap, (unsigned)yv.y, sse);
                        const unsigned f = resize_dword<decltype(mode)::value>(
                            wd + __umul24(((unsigned)zv.x & 0xFFFFu) - wy0, ws),
                            wd + __umul24(((unsigned)zv.x >> 16) - wy0, ws), shb, sel, tap, (unsigned)zv.y, sse);
                        emit(ey, d);
                        if (ez != ey) emit(ez, f);
                    }
                };
                if (rmode == 1) rows(ModeTag<1>{});
                else if (rmode == 0) rows(ModeTag<0>{});
                else rows(ModeTag<2>{});
            } else {
                for (int ey = r0; ey < nrows; ey += rstep) {
                    const int2 yv = s_row[k & 1][ey];
                    emit(ey, resize4((const uint8_t*)src, __umul24(((unsigned)yv.x & 0xFFFFu) - wy0, 4 * ws),
                                     __umul24(((unsigned)yv.x >> 16) - wy0, 4 * ws), sxk, nxk, tap, yv.y, sse));
                }
            }
        }
        if (k < m) {
            if (tid < ORB_CH_ROWS) s_row[(k + 1) & 1][tid] = make_int2((int)yt.x, (int)yt.y);
            __syncthreads();
        }
    }
}

// level < 0: the tiles of every level whose tile height is TH.
template <int TH>
__global__ __launch_bounds__(256) void level_kernel(const ImageJob* __restrict__ jobs,
                                                    const RunTable* __restrict__ rt, int level)
{
    __shared__ __align__(16) unsigned pxw[(TH + 2 * LT_HALO) + 1][LP_WD];   // level pixels, tile + 4-px halo (and what
                                                                            // the blur's 32-byte windows reach past)
    __shared__ unsigned mmw[(TH + 2)][LP_WD];         // FAST strength, tile + 1-px ring
    __shared__ unsigned short queue[(TH + 2) * (LT_W + 2)];   // FAST candidates
    __shared__ unsigned kloc[LK_CAP];            // tile-local keypoints: ly | lx | score | passes
    __shared__ int s_qn, s_nq, s_kn, s_base;
    __shared__ int s_col[LT_W], s_row[TH];      // FAST cell of each tile column / row, edge flags
    const uint8_t* px = (const uint8_t*)pxw;
    uint8_t* mm = (uint8_t*)mmw;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    // Every wave finds its tile itself (uniform scalar loads), so the first
    // barrier comes only after the tile's memory reads have been issued; the
    // counters cleared here are first used after that barrier.
    int blk = xcd_block(blockIdx.x, gridDim.x);
    if (level < 0) {
        const int* starts = rt->all_start[TH == 16 ? 1 : 0];
        level = 0;
        while (blk >= starts[level + 1]) level++;
        blk -= starts[level];
    }
    const int tpj = rt->tiles_per_job[level];
    // (Divisions by reciprocals: each of the 4 wavefronts does this, and scalar
    // instructions count: 50 more of them were 24 us of 463 in a batch, and these
    // reciprocals, with the interior tiles' own loads and stores, 22 fewer.)
    int job, t;
    if (tpj > 0) {
        job = (int)__umulhi(2u * (unsigned)blk, rt->tiles_rcp[level]);
        t = blk - job * tpj;
    } else {
        job = find_segment(rt->tile_start[level], rt->njobs, blk);
        t = blk - rt->tile_start[level][job];
    }
    if (tid == 0) {
        s_qn = 0;
        s_nq = 0;
        s_kn = 0;
    }
    const ImageJob& J = jobs[job];
    const LevelJob& L = J.lv[level];
    const int trow = (int)__umulhi(2u * (unsigned)t, L.txrcp);
    const int tx0 = (t - trow * L.tiles_x) * LT_W;
    const int ty0 = trow * TH;
    const int w = L.w, h = L.h, pitch = L.pitch;
    const bool interior = tx0 >= LT_HALO && tx0 + LT_W + LT_HALO <= w && ty0 >= LT_HALO &&
                          ty0 + TH + LT_HALO <= h;

    // FAST detection area of the level.
    const int ax0 = ORB_EDGE, ay0 = ORB_EDGE;
    const int ax1 = min(ORB_EDGE + L.nCols * L.wCell, L.maxBorderX - 3);
    const int ay1 = min(ORB_EDGE + L.nRows * L.hCell, L.maxBorderY - 3);
    // Per tile column: its FAST cell column cj, and whether the pixels left
    // and right of it fall outside that cell's window (bits 16, 17); rows
    // likewise.  Built while the tile's first reads are in flight; read
    // after later barriers.
    auto cell_tables = [&]() {
        if (tid < LT_W + TH) {
            const bool isc = tid < LT_W;
            const int z = isc ? tx0 + tid : ty0 + (tid - LT_W);
            const int cs = isc ? L.wCell : L.hCell, a0 = isc ? ax0 : ay0, a1 = isc ? ax1 : ay1;
            const int cz = (int)__umulhi((unsigned)max(z - ORB_EDGE, 0), isc ? L.wrcp : L.hrcp);   // / cs
            const int c0 = max(ORB_EDGE + cz * cs, a0), c1 = min(ORB_EDGE + (cz + 1) * cs, a1);
            const int info = cz | ((z - 1 < c0) << 16) | ((z + 1 >= c1) << 17);
            if (isc) s_col[tid] = info;
            else s_row[tid - LT_W] = info;
        }
    };

    // ---- 1. pixels with halo, one dword (4 columns) per slot: 720 (or 432)
    // dwords, 3 per thread, read before any wait (indexes past the end repeat
    // the last dword).  A border tile reads reflected rows (REFLECT_101), and
    // bytewise the dwords that reach past a level edge, as far as the halo is
    // used (3 pixels).
    {
        const uint8_t* src = level == 0 ? J.src : L.lvl;
        const int sp = level == 0 ? J.src_pitch : pitch;
        unsigned d[3];
        static_assert(256 == 14 * LP_WD + 4, "the next dword is 14 rows and 4 dwords on");
        int ey = tid / LP_WD, ex = tid - ey * LP_WD;
        auto next = [&]() {
            const int past = ex + 4 >= LP_WD ? 1 : 0;
            ey = min(ey + 14 + past, TH + 2 * LT_HALO - 1);
            ex = ex + 4 - past * LP_WD;
        };
        if (interior && (sp & 3) == 0) {
            const uint8_t* s0 = src + (unsigned)((ty0 - LT_HALO) * sp + tx0 - LT_HALO);
#pragma unroll
            for (int k = 0; k < 3; k++) {
                if (k) next();
                d[k] = gload4(s0 + (unsigned)(__umul24(ey, sp) + 4 * ex));
            }
        } else {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                if (k) next();
                const int x = tx0 - LT_HALO + ex * 4, y = reflect101(ty0 - LT_HALO + ey, h);
                if (x >= 0 && x + 3 < w) {
                    d[k] = gload4u(src + (unsigned)(y * sp + x));
                } else {
                    d[k] = 0;
                    const uint8_t* r = src + (size_t)y * sp;
                    if (x < w + LT_HALO) {
#pragma unroll
                        for (int q = 0; q < 4; q++) d[k] |= (unsigned)gload1(r + reflect101(x + q, w)) << (8 * q);
                    }
                }
            }
        }
        cell_tables();
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const int e = tid + 256 * k;
            if (e < (TH + 2 * LT_HALO) * LP_WD) (&pxw[0][0])[e] = d[k];
        }
    }
    __syncthreads();

    // ---- 2. the level (copied out) and its 7x7 blur
    const int gc = tid & 15;                      // 4-column group of the tile
    // Level 0 copied out when the input is not level 0 itself (levels >= 1
    // are the pyramid kernel's).
    if (level == 0 && J.src != L.lvl) {
        for (int r = tid >> 4; r < TH; r += 16) {
            const int y = ty0 + r, x0 = tx0 + 4 * gc;
            if (y >= h) continue;
            const unsigned d = pxw[r + LT_HALO][gc + 1];
            uint8_t* dst = L.lvl + (unsigned)(y * pitch + x0);
            if (x0 + 3 < w) {
                gstore4(dst, d);
            } else {
                for (int k = 0; k < 4; k++)
                    if (x0 + k < w) dst[k] = (uint8_t)(d >> (8 * k));
            }
        }
    }
    // The blur: a wavefront takes 16 columns.  Row sums of 16 rows at a time
    // are pixels (as signed bytes) times the column band; they fit 16 bits,
    // and a lane then holds 4 rows of one column, which is where the second
    // product takes its k from: signed high and low bytes times the row band,
    // laid out so that a lane ends with 4 columns of one row.  Rows and bytes
    // past the tile's halo meet zero taps.  As two passes of v_dot4 and 24-bit
    // multiplies through LDS it was 200 vector instructions a wavefront and two
    // barriers, and the kernel is bound by those: 128 images of 1241 x 376 500 us
    // so, 460 with the matrix units; 64 of four sizes 280 and 256.
    {
        const int g = lane >> 4, n = lane & 15, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
        const long colband = __builtin_bit_cast(long, c_band[0][lane]), rowband = __builtin_bit_cast(long, c_band[1][lane]);
        const int cb = c_bandsum[0], rs = c_bandsum[1];
        const orb_v4i bias0 = {cb, cb, cb, cb}, bias1 = {rs, rs, rs, rs}, none = {0, 0, 0, 0};
        unsigned lo[TH / 16 + 1], hi[TH / 16 + 1];
#pragma unroll
        for (int t = 0; t <= TH / 16; t++) {
            uint2 a = *(const uint2*)&pxw[min(16 * t + n + 1, TH + 2 * LT_HALO - 1)][4 * wv + 2 * g];
            a.x ^= 0x80808080u;
            a.y ^= 0x80808080u;
            const orb_v4i sums =                   // row sum - 32768
                __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, a), colband, bias0, 0, 0, 0);
            const unsigned p01 = __builtin_amdgcn_perm((unsigned)sums[1], (unsigned)sums[0], 0x05010400u);
            const unsigned p23 = __builtin_amdgcn_perm((unsigned)sums[3], (unsigned)sums[2], 0x05010400u);
            lo[t] = __builtin_amdgcn_perm(p23, p01, 0x05040100u) ^ 0x80808080u;
            hi[t] = __builtin_amdgcn_perm(p23, p01, 0x07060302u);
        }
        // Column rounding: columns < bs_end as OpenCV's SSE2 column kernel
        // (SymmColumnVec_32s8u: the taps as floats k / 2^16, the sum rounded
        // half to even, which for these exact sums is (acc + 0x7FFF + bit 16
        // of acc) >> 16), the others as its scalar one ((acc + 2^15) >> 16).
        // rb: how many bits of acc's bit 16 count (1 or 0).
        const int x0 = tx0 + 16 * wv + 4 * g;
        unsigned rb[4];
#pragma unroll
        for (int k = 0; k < 4; k++) rb[k] = x0 + k < L.bs_end ? 1u : 0u;
#pragma unroll
        for (int t = 0; t < TH / 16; t++) {
            const orb_v4i high = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                __builtin_bit_cast(long, make_uint2(hi[t], hi[t + 1])), rowband, none, 0, 0, 0);
            const orb_v4i low = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                __builtin_bit_cast(long, make_uint2(lo[t], lo[t + 1])), rowband, bias1, 0, 0, 0);
            unsigned v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const unsigned acc = ((unsigned)high[k] << 8) + (unsigned)low[k];
                v[k] = acc + __builtin_amdgcn_ubfe(acc, 16, rb[k]) + (0x8000u - rb[k]);
            }
            // >> 16, clamped to 255 two at a time, and the four bytes gathered
            const orb_us2 top = {255, 255};
            const unsigned v01 = __builtin_bit_cast(unsigned, __builtin_elementwise_min(
                __builtin_bit_cast(orb_us2, __builtin_amdgcn_perm(v[1], v[0], 0x07060302u)), top));
            const unsigned v23 = __builtin_bit_cast(unsigned, __builtin_elementwise_min(
                __builtin_bit_cast(orb_us2, __builtin_amdgcn_perm(v[3], v[2], 0x07060302u)), top));
            const unsigned out = __builtin_amdgcn_perm(v23, v01, 0x06040200u);
            const int y = ty0 + 16 * t + n;
            uint8_t* db = L.blur + (unsigned)(y * pitch + x0);
            if (interior) {
                gstore4(db, out);
            } else if (y < h) {
                if (x0 + 3 < w) {
                    gstore4(db, out);
                } else {
                    for (int k = 0; k < 4; k++)
                        if (x0 + k < w) db[k] = (uint8_t)(out >> (8 * k));
                }
            }
        }
    }

    // ---- 3. FAST strength on the tile plus a 1-px ring, detection areas
    // only.  The cardinal pre-test runs on 12-pixel groups (two pixels per
    // 16-bit lane pair); survivors are compacted, then scored exactly.
    const int tA = min(max(J.iniTh, 0), 255), tB = min(max(J.minTh, 0), 255);
    const int tmin = min(tA, tB);
    const unsigned t2 = (unsigned)tmin | ((unsigned)tmin << 16);
    // tile plus its 1-px ring wholly inside the detection area
    const bool tile_in = tx0 - 1 >= ax0 && tx0 + LT_W < ax1 && ty0 - 1 >= ay0 && ty0 + TH < ay1;
    // Lanes: rows tile -1..32 and 12-column groups g = 0..5 (px dwords 3g ..
    // 3g + 2, tile columns 12g - 4 .. 12g + 7): 204 lanes, one pass.  Group 0
    // only contributes its pixels 3.. (tile columns -1..) and group 5 its
    // pixels ..8 (columns ..64): the 1-px ring.  Their missing neighbour
    // dwords (columns -8 and 68 onwards) feed only the bytes masked off.
    static_assert((TH + 2) * 6 <= 256, "one pre-test pass");
    static_assert(LP_WD == 18, "6 lanes of 3 dwords cover a strength-map row");
    {
        unsigned cand = 0u;                       // bit k: pixel k of the group
        int my = 0, g = 0;
        if (tid < (TH + 2) * 6) {
            my = tid / 6;
            g = tid - my * 6;
            const int y = ty0 - 1 + my;
            const int py = my + 3;                // px row of tile row y
            const int x = tx0 + 12 * g - 4;
            const unsigned* vr = &pxw[py][3 * g];
            const unsigned* ur = &pxw[py - 3][3 * g];
            const unsigned* dr = &pxw[py + 3][3 * g];
            // The lanes tile the strength map exactly (34 rows x 18 dwords):
            // each clears its 3 dwords; candidates get their strength below.
            mmw[my][3 * g] = 0u;
            mmw[my][3 * g + 1] = 0u;
            mmw[my][3 * g + 2] = 0u;
            const unsigned Vx = vr[0], Vy = vr[1], Vz = vr[2];
            const unsigned Lw = g > 0 ? vr[-1] : 0u;
            const unsigned Rw = g < 5 ? vr[3] : 0u;
            // Even / odd pixels of each dword in 16-bit lanes (lo / hi =
            // pixels 0, 2 / 1, 3 of the dword); the neighbours 3 columns
            // right (p4) and left (p12) are byte selections of the row.
            const unsigned Vxl = lo_bytes(Vx), Vxh = hi_bytes(Vx), Vyl = lo_bytes(Vy), Vyh = hi_bytes(Vy);
            const unsigned Vzl = lo_bytes(Vz), Vzh = hi_bytes(Vz);
            const unsigned m02a = fast_maybe2(Vxl, lo_bytes(dr[0]), __builtin_amdgcn_perm(Vy, Vx, 0x0C050C03u),
                                              lo_bytes(ur[0]), hi_bytes(Lw), t2);        // columns 0, 2
            const unsigned m13a = fast_maybe2(Vxh, hi_bytes(dr[0]), Vyl, hi_bytes(ur[0]),
                                              __builtin_amdgcn_perm(Vx, Lw, 0x0C040C02u), t2);   // 1, 3
            const unsigned m02b = fast_maybe2(Vyl, lo_bytes(dr[1]), __builtin_amdgcn_perm(Vz, Vy, 0x0C050C03u),
                                              lo_bytes(ur[1]), Vxh, t2);                 // 4, 6
            const unsigned m13b = fast_maybe2(Vyh, hi_bytes(dr[1]), Vzl, hi_bytes(ur[1]),
                                              __builtin_amdgcn_perm(Vy, Vx, 0x0C040C02u), t2);   // 5, 7
            const unsigned m02c = fast_maybe2(Vzl, lo_bytes(dr[2]), __builtin_amdgcn_perm(Rw, Vz, 0x0C050C03u),
                                              lo_bytes(ur[2]), Vyh, t2);                 // 8, 10
            const unsigned m13c = fast_maybe2(Vzh, hi_bytes(dr[2]), lo_bytes(Rw), hi_bytes(ur[2]),
                                              __builtin_amdgcn_perm(Vz, Vy, 0x0C040C02u), t2);   // 9, 11
            // pixels k in [klo, khi): detection area, and the ring rule
            unsigned mask;
            if (tile_in) {
                mask = g == 0 ? 0xFF8u : (g == 5 ? 0x1FFu : 0xFFFu);
            } else {
                const int klo = min(max(max(ax0 - x, g == 0 ? 3 : 0), 0), 12);
                const int khi = max(min(min(ax1 - x, g == 5 ? 9 : 12), 12), 0);
                const bool yin = y >= ay0 && y < ay1;
                mask = (yin && klo < khi) ? ((1u << khi) - (1u << klo)) : 0u;
            }
            // each 16-bit lane clamped to 0 / 1: pixel k's bit at k (k = 0, 1,
            // 4, 5, 8, 9) or k + 14 (k = 2, 3, 6, 7, 10, 11)
            // (1 | 1 << 16 hidden from the optimiser, which otherwise turns
            // the clamp into per-lane compares and selects)
            unsigned one2 = 0x00010001u;
            asm volatile("" : "+s"(one2));
            const orb_us2 one = __builtin_bit_cast(orb_us2, one2);
#define ORB_BIT01(m) __builtin_bit_cast(unsigned, __builtin_elementwise_min(__builtin_bit_cast(orb_us2, m), one))
            const unsigned x01 = ORB_BIT01(m02a) | (ORB_BIT01(m13a) << 1) | (ORB_BIT01(m02b) << 4) |
                                 (ORB_BIT01(m13b) << 5) | (ORB_BIT01(m02c) << 8) | (ORB_BIT01(m13c) << 9);
#undef ORB_BIT01
            cand = (x01 | (x01 >> 14)) & mask;
        }
        // Append: the wave's exclusive prefix of the per-lane counts (0..12)
        // from four ballots of the count's bits, one LDS atomic per wave.
        const int cnt = __popc(cand);
        const unsigned long long b0 = __ballot(cnt & 1), b1 = __ballot(cnt & 2), b2 = __ballot(cnt & 4),
                                 b3 = __ballot(cnt & 8);
        const int tot = __popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2) + 8 * __popcll(b3);
        if (tot) {
            int base = 0;
            if (lane == 0) base = atomicAdd(&s_qn, tot);
            base = __builtin_amdgcn_readfirstlane(base);     // every lane is active here
            int pos = base + lanes_below(b0) + 2 * lanes_below(b1) + 4 * lanes_below(b2) + 8 * lanes_below(b3);
            // queue entry: m-row << 8 | byte column in mmw (tile col + 4)
            const unsigned ebase = ((unsigned)my << 8) | (unsigned)(12 * g);
            for (unsigned m = cand; m; m &= m - 1)
                queue[pos++] = (unsigned short)(ebase + (unsigned)__builtin_ctz(m));
        }
    }
    __syncthreads();
    // Exact strengths of the queued pixels, two per thread before one barrier.
    // Pixels of the tile proper that beat the lower threshold are compacted
    // again, in place (a slot is only rewritten after the barrier that ends
    // the reads of its chunk of 512), so that suppression runs on dense lanes.
    const int qn = s_qn;
    for (int q0 = 0; q0 < qn; q0 += 512) {
        int e[2] = {0, 0};
        bool keep[2] = {false, false};
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int q = q0 + 256 * h + tid;
            if (q < qn) {
                e[h] = queue[q];
                const int my = e[h] >> 8, col = e[h] & 255;
                const int sv = fast_strength(px + (my + 3) * LP_W + col, LP_W);
                mm[my * LP_W + col] = (uint8_t)sv;
                keep[h] = sv > tmin && my >= 1 && my <= TH && col >= 4 && col < 4 + LT_W;
            }
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const unsigned long long bal = __ballot(keep[h]);
            if (bal) {
                int base = 0;
                if (lane == 0) base = atomicAdd(&s_nq, __popcll(bal));
                base = __builtin_amdgcn_readfirstlane(base);     // every lane is active here
                if (keep[h]) queue[base + lanes_below(bal)] = (unsigned short)e[h];
            }
        }
    }
    __syncthreads();

    // ---- 4. per-cell non-max suppression at both thresholds.  A neighbour's
    // score at threshold t is (m > t ? m - 1 : 0) for its strength m, 0 outside
    // the cell's window; it grows with m, so the largest neighbour score is
    // the score of the largest in-window neighbour strength M.  The pixel is
    // kept at t iff mc > t and mc - 1 > score(M) (which is >= 0, so this also
    // beats the out-of-window zeros).
    const int nq = s_nq;
    for (int q0 = 0; q0 < nq; q0 += 256) {
        const int q = q0 + tid;
        bool keepA = false, keepB = false;
        unsigned loc = 0u;
        if (q < nq) {
            const int e = queue[q];
            const int ly = (e >> 8) - 1, lx = (e & 255) - 4;
            const uint8_t* mrow = mm + (ly + 1) * LP_W + (lx + 4);
            const int mc = mrow[0];
            const int colv = s_col[lx], rowv = s_row[ly];
            int M = 0;
#pragma unroll
            for (int n = 0; n < 9; n++) {
                if (n == 4) continue;
                const int dx = n % 3 - 1, dy = n / 3 - 1;
                const bool out = (dx < 0 && (colv & 0x10000)) || (dx > 0 && (colv & 0x20000)) ||
                                 (dy < 0 && (rowv & 0x10000)) || (dy > 0 && (rowv & 0x20000));
                const int mq = mrow[dy * LP_W + dx];
                M = max(M, out ? 0 : mq);
            }
            keepA = mc > tA && mc - 1 > (M > tA ? M - 1 : 0);
            keepB = mc > tB && mc - 1 > (M > tB ? M - 1 : 0);
            loc = ((unsigned)ly << 6) | (unsigned)lx | ((unsigned)mc << 11);
            if (keepA) gstore1(L.cellflag + (rowv & 0xFFFF) * L.nCols + (colv & 0xFFFF), 1);
        }
        // Append, one entry for both passes: the wave's prefix from a ballot,
        // one LDS atomic per wave.
        const bool keep = keepA || keepB;
        const unsigned long long bal = __ballot(keep);
        if (bal) {
            int base = 0;
            if (lane == 0) base = atomicAdd(&s_kn, __popcll(bal));
            base = __builtin_amdgcn_readfirstlane(base);     // every lane is active here
            const int pos = base + lanes_below(bal);
            if (keep && pos < LK_CAP) kloc[pos] = loc | (keepA ? 1u << 19 : 0u) | (keepB ? 1u << 20 : 0u);
        }
    }
    __syncthreads();

    // ---- 5. append the tile's candidates to one of the level's lists as
    // (score << 32 | cell row, cell col, y, x in cell) | passes
    const int kn = s_kn;
    if (kn == 0) return;
    if (tid == 0) {
        s_base = atomicAdd(L.segs + t % ORB_SEGS * ORB_SEG_STRIDE, kn);
        if (kn > LK_CAP || s_base + kn > L.seg_cap) atomicOr(&J.counters[ORB_CNT_ERR], ORB_ERR_KEYS);
    }
    __syncthreads();
    const int base = s_base;
    unsigned long long* keys = L.keys + (size_t)(t % ORB_SEGS) * L.seg_cap;
    for (int i = tid; i < min(kn, LK_CAP); i += 256) {
        if (base + i >= L.seg_cap) break;
        const unsigned loc = kloc[i];
        const int x = tx0 + (int)(loc & 63u), y = ty0 + (int)((loc >> 6) & 31u);
        const int mc = (int)((loc >> 11) & 255u);
        const int cj = s_col[loc & 63u] & 0xFFFF, ci = s_row[(loc >> 6) & 31u] & 0xFFFF;
        const unsigned xl = (unsigned)(x - (ORB_MIN_BORDER + cj * L.wCell));
        const unsigned yl = (unsigned)(y - (ORB_MIN_BORDER + ci * L.hCell));
        const unsigned ok = ((unsigned)ci << 20) | ((unsigned)cj << 12) | (yl << 6) | xl;
        unsigned long long key = ((unsigned long long)(unsigned)(mc - 1) << 32) | ok;
        key |= (unsigned long long)((loc >> 19) & 3u) << 40;         // ORB_KEY_INI, ORB_KEY_MIN
        gstore8(keys + base + i, key);
    }
}

// ================================================================ octree
// DistributeOctTree (ORBextractor.cc:688-1033) on one workgroup per level.
//
// The reference keeps a std::list of nodes.  Phase 1 repeats full passes,
// splitting every node with more than one key and pushing its non-empty
// children to the list front (n1..n4, so they read n4,n3,n2,n1); phase 2
// sorts the expandable nodes by (size, address) and splits from the largest
// until the quota is reached.  Here the list is an array in LDS; each candidate
// carries the index of the list node that holds it.  octree_fast finds the
// list at the end of phase 1 at once; octree_general, for the candidate sets
// it does not reach, rebuilds the list each pass with prefix sums.  Node
// order, membership and retained keys are exactly the list's.  Ties in the phase-2 sort are broken by creation order
// (newer = larger), the oracle's fixed stand-in for the heap address.
#define OCT_T 1024
static_assert(OCT_T == 64 * ORB_SEGS, "a wavefront per candidate list");
#define OCT_REG 4                    // general form: candidates per thread held in registers
#define OCT_D ORB_OCT_D
#define OCT_KEYS 8192                // fast form: candidates held in LDS (the others in global memory)
#define OCT_CELLS 2048               // fast form: cells of the depth that ends phase 1
#define OCT_FLAGS 4096               // fast form: FAST cells whose flags are held in LDS
// Words of the occupancy bitmaps of depths OCT_D .. 0 for n roots, one after
// another: n * 4^d cells at depth d.
#define OCT_WORDS(n) (170 * (n) + ((n) + 1) / 2 + ((n) + 7) / 8 + 1)

struct OctGeneral {
    int rx[2][ORB_LIST_CAP];     // x0 | x1 << 16
    int ry[2][ORB_LIST_CAP];     // y0 | y1 << 16
    int cnt[2][ORB_LIST_CAP];
    int seq[2][ORB_LIST_CAP];
    int cc[ORB_LIST_CAP][4];
    short map[ORB_LIST_CAP][4];
    short keep[ORB_LIST_CAP];
    unsigned long long sortk[ORB_LIST_CAP];
    unsigned long long best[ORB_LIST_CAP];
    int scan[2][OCT_T / 64];
    int vars[8];
};

struct OctFast {
    unsigned key[OCT_KEYS];      // place at depth OCT_D | list node << 16
    union {
        unsigned bm[2][OCT_WORDS(ORB_MAX_ROOTS)];   // occupied cells; cells of two or more keys
        struct {
            int4 cc[ORB_LIST_CAP];       // keys per quadrant of a node
            unsigned at[ORB_LIST_CAP];   // where the round puts a node or its children
        };
    };
    union {
        int cell[OCT_CELLS];     // list node of each cell of the depth that ends phase 1
        unsigned long long best[ORB_LIST_CAP];
    };
    union {
        uint8_t flag[OCT_FLAGS];
        unsigned sortk[ORB_LIST_CAP];
    };
    unsigned short order[ORB_LIST_CAP];
    unsigned done[ORB_LIST_CAP / 32];   // nodes split in this round
    int scan[2][OCT_T / 64];
    int na[OCT_D + 1], nm[OCT_D + 1];   // set bits per depth
    int nkeys, nexp, end, deep, p1, size, cp;
};

// First word of depth d's bitmap (n roots).
__device__ __forceinline__ int oct_word0(int d, int n)
{
    const int w = d == 6 ? 0 : (d == 5 ? 128 : (d == 4 ? 160 : (d == 3 ? 168 : 170)));
    return w * n + (d < 2 ? (n + 1) / 2 : 0) + (d < 1 ? (n + 7) / 8 : 0);
}

// LDS written by this wavefront is read by its other lanes next.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Inclusive scan over the wavefront by DPP (rows of 16, then the row totals).
__device__ __forceinline__ int wave_scan(int v)
{
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);   // row_shr:1
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);   // row_shr:2
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);   // row_shr:4
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);   // row_shr:8
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);   // row_bcast:15 to rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);   // row_bcast:31 to rows 2 and 3
    return v;
}

// Exclusive scan over the workgroup, and the total: one barrier.  Two scans
// in a row use the two halves of sh in turn (`half`), so that a scan's writes
// never meet the reads of the one before.
__device__ __forceinline__ int block_scan(int v, int (*sh)[OCT_T / 64], int& half, int* total)
{
    static_assert(OCT_T / 64 == 16, "a row of 16 lanes scans the wavefronts' totals");
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = wave_scan(v);
    int* h = sh[half];
    half ^= 1;
    if (lane == 63) h[wid] = x;
    __syncthreads();
    int t = h[lane & 15];
    t += __builtin_amdgcn_update_dpp(0, t, 0x111, 0xF, 0xF, false);
    t += __builtin_amdgcn_update_dpp(0, t, 0x112, 0xF, 0xF, false);
    t += __builtin_amdgcn_update_dpp(0, t, 0x114, 0xF, 0xF, false);
    t += __builtin_amdgcn_update_dpp(0, t, 0x118, 0xF, 0xF, false);
    *total = __builtin_amdgcn_readlane(t, 15);
    const int below = wid > 0 ? __builtin_amdgcn_readlane(t, wid > 0 ? wid - 1 : 0) : 0;
    return below + x - v;
}

__device__ __forceinline__ void key_xy(unsigned long long key, int wCell, int hCell, int* x, int* y)
{
    const unsigned ok = (unsigned)key;
    const int xl = ok & 63, yl = (ok >> 6) & 63, j = (ok >> 12) & 255, i = (ok >> 20) & 255;
    *x = j * wCell + xl;
    *y = i * hCell + yl;
}

__device__ __forceinline__ int quad_of(int rx, int ry, int x, int y)
{
    const int x0 = rx & 0xFFFF, x1 = rx >> 16, y0 = ry & 0xFFFF, y1 = ry >> 16;
    const int mx = x0 + ((x1 - x0 + 1) >> 1), my = y0 + ((y1 - y0 + 1) >> 1);
    return (x < mx ? 0 : 1) + (y < my ? 0 : 2);
}

__device__ __forceinline__ void child_rect(int rx, int ry, int q, int* crx, int* cry)
{
    const int x0 = rx & 0xFFFF, x1 = rx >> 16, y0 = ry & 0xFFFF, y1 = ry >> 16;
    const int mx = x0 + ((x1 - x0 + 1) >> 1), my = y0 + ((y1 - y0 + 1) >> 1);
    const int cx0 = (q & 1) ? mx : x0, cx1 = (q & 1) ? x1 : mx;
    const int cy0 = (q & 2) ? my : y0, cy1 = (q & 2) ? y1 : my;
    *crx = cx0 | (cx1 << 16);
    *cry = cy0 | (cy1 << 16);
}

// The fast form.  A key's path through the quadtree depends on its position
// alone, so all of phase 1 can be found at once:
//   - A cell's place among its depth's cells in list order is a number that
//     follows from its path: a pass pushes the children of the nodes it
//     visits in list order to the front, so with o_0 = root and M_d = roots *
//     4^d, o_d = M_d - 1 - (4 o_{d-1} + quadrant): the quadrants' digits, every
//     other one turned around.  A key's place at depth OCT_D comes from two
//     tables (its x and its y); its places above are shifts of that.
//   - Every key marks its depth-OCT_D cell in a bitmap, and in a second one
//     if the cell was marked; the shallower depths' bitmaps follow by nibbles.
//     The list after pass p has as many nodes as depth p has occupied cells,
//     and as many to expand as cells of two or more keys: that decides the
//     pass p1 that ends phase 1.
//   - Its list is the depth-p1 cells by o_p1, then the single-key cells of
//     depth p1 - 1 whose parent was split, by their o, and so on to the
//     roots: marking every cell's node in that order and counting the marks
//     below it numbers the nodes, per cell of depth p1, not per key.
// Phase 2 then needs only the keys per quadrant of each node: the nodes it
// may split are those of the last pass, all of one depth, and the reference's
// (size, newest first) order among them is (size, list position).
// Returns false where it does not reach: phase 1 beyond depth OCT_D - 1 or
// OCT_CELLS cells, a split of a depth-OCT_D cell (candidates in small
// clusters).
// Bound: latency (barriers, LDS round trips, and 16 cycles an instruction
// where all 16 wavefronts run it).  640x480 with 1000 features 14.5 us (27 pass
// by pass), 1280x720 with 2000 25 us (55), 128 images of 1241x376 63 us (105),
// 64 of four sizes 43 us (95).
__device__ __forceinline__ bool octree_fast(OctFast& S, const LevelJob& L, int level, int* ctr)
{
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    // this wavefront's candidate list
    const int K0 = min(L.segs[wv * ORB_SEG_STRIDE], L.seg_cap);
    const unsigned long long* list = L.keys + (size_t)wv * L.seg_cap;
    const int N = L.quota, n = L.nIni, nCols = L.nCols, ncells = L.ncells;
    const int wC = L.wCell, hC = L.hCell;
    const int nwords = OCT_WORDS(n);
    int half = 0;
    // A candidate's place | node << 16: in LDS, or in global memory past OCT_KEYS.
    auto put = [&](int k, unsigned v) {
        if (k < OCT_KEYS) S.key[k] = v;
        else gstore4((uint8_t*)(L.node + k), v);
    };
    auto get = [&](int k) { return k < OCT_KEYS ? S.key[k] : gload4((const uint8_t*)(L.node + k)); };

    // ---- the per-cell retry (ORBextractor.cc:1111-1124): a cell keeps its
    // iniThFAST candidates when it has any, else its minThFAST candidates.
    // The survivors' places go to LDS, the survivors to keys2 (in any order:
    // the level kernels append them in none, and the result depends on the
    // set alone).
    unsigned long long key[4];
#pragma unroll
    for (int m = 0; m < 4; m++) key[m] = gload8u64(list + min(lane + 64 * m, max(K0 - 1, 0)));
    const bool lds_flags = ncells <= OCT_FLAGS;
    if (lds_flags)
        for (int i = tid; i < ncells; i += OCT_T) S.flag[i] = gload1(L.cellflag + i);
    for (int i = tid; i < nwords; i += OCT_T) S.bm[0][i] = S.bm[1][i] = 0u;
    if (tid <= OCT_D) S.na[tid] = S.nm[tid] = 0;
    if (tid == 0) S.nkeys = S.deep = 0;
    __syncthreads();
    for (int c0 = 0; c0 < K0; c0 += 4 * 64) {
        unsigned o[4];
        unsigned long long k[4];
        int cnt = 0;
        bool v[4];
#pragma unroll
        for (int m = 0; m < 4; m++) {
            k[m] = key[m];
            const unsigned ok = (unsigned)k[m];
            const unsigned xl = ok & 63, yl = (ok >> 6) & 63, j = (ok >> 12) & 255, i = (ok >> 20) & 255;
            o[m] = (unsigned)(L.octx[__umul24(j, wC) + xl] ^ L.octy[__umul24(i, hC) + yl]);
            const unsigned c = __umul24(i, nCols) + j;
            const int f = lds_flags ? S.flag[c] : gload1(L.cellflag + c);
            v[m] = c0 + lane + 64 * m < K0 && (k[m] & (f ? ORB_KEY_INI : ORB_KEY_MIN));
            cnt += v[m] ? 1 : 0;
        }
        if (c0 + 4 * 64 < K0) {
#pragma unroll
            for (int m = 0; m < 4; m++) key[m] = gload8u64(list + min(c0 + 4 * 64 + lane + 64 * m, K0 - 1));
        }
        const int inc = wave_scan(cnt);
        int base = 0;
        if (lane == 63 && inc) base = atomicAdd(&S.nkeys, inc);
        int pos = __builtin_amdgcn_readlane(base, 63) + inc - cnt;
#pragma unroll
        for (int m = 0; m < 4; m++)
            if (v[m]) {
                put(pos, o[m]);
                gstore8(L.keys2 + pos++, k[m] & ORB_KEY_RANK);
                const unsigned bit = 1u << (o[m] & 31);
                if (atomicOr(&S.bm[0][o[m] >> 5], bit) & bit) atomicOr(&S.bm[1][o[m] >> 5], bit);
            }
    }
    __syncthreads();
    const int K = S.nkeys;

    // ---- occupancy of the shallower depths: cell o's children are nibble
    // M - 1 - o of the next depth
    auto reduce = [&](int d, int o) {
        const int M = n << (2 * d), w0 = oct_word0(d, n), wc = oct_word0(d + 1, n);
        bool occ = false, multi = false;
        if (o < M) {
            const int c = M - 1 - o;
            const unsigned ca = (S.bm[0][wc + (c >> 3)] >> (4 * (c & 7))) & 15u;
            const unsigned cm = (S.bm[1][wc + (c >> 3)] >> (4 * (c & 7))) & 15u;
            occ = ca != 0;
            multi = cm != 0 || (ca & (ca - 1)) != 0;
        }
        const unsigned long long ba = __ballot(occ), bb = __ballot(multi);
        const int w = (o >> 5) & ~1;             // the wavefront's two words
        if (lane < 2 && 32 * (w + lane) < M) {
            S.bm[0][w0 + w + lane] = (unsigned)(ba >> (32 * lane));
            S.bm[1][w0 + w + lane] = (unsigned)(bb >> (32 * lane));
        }
        if (lane == 0 && ba) {
            atomicAdd(&S.na[d], __popcll(ba));
            atomicAdd(&S.nm[d], __popcll(bb));
        }
    };
    for (int o = tid; o - lane < n << 10; o += OCT_T) reduce(5, o);
    __syncthreads();
    for (int o = tid; o - lane < n << 8; o += OCT_T) reduce(4, o);
    __syncthreads();
    if (wv == 0) {                               // the others wait at the barrier below
        for (int d = 3; d >= 0; d--) {
            for (int o = lane; o - lane < n << (2 * d); o += 64) reduce(d, o);
            wave_lds_sync();
        }
        // the pass that ends phase 1 (ORBextractor.cc:779-893), lane p = pass p
        const int p = min(lane, OCT_D), size = S.na[p], prev = S.na[max(p - 1, 0)], nexp = S.nm[p];
        const bool last = size >= N || size == prev;
        const unsigned long long ends = __ballot(lane >= 1 && lane < OCT_D &&
                                                 (last || size + 3 * nexp > N || size > ORB_LIST_CAP));
        const int p1 = ends ? __ffsll((long long)ends) - 1 : 0;
        if (lane == p1) {
            S.p1 = p1;
            S.size = size;
            S.end = last ? 1 : 0;
        }
    }
    __syncthreads();
    const int p1 = S.p1;
    int size = S.size;
    const int M = n << (2 * p1);
    if (p1 == 0 || M > OCT_CELLS || size > ORB_LIST_CAP) return false;
    bool more = !S.end;

    // ---- the list after pass p1: every occupied depth-p1 cell's node, the
    // shallowest cell of one key above it or the cell itself, as depth << 17 |
    // place.  Cells are numbered as shifts of the depth-OCT_D place: the place
    // at depth p1, turned around where OCT_D - p1 is odd.
    const int sh = 2 * (OCT_D - p1);
    const bool turn = p1 & 1;
    const int wfirst = oct_word0(p1, n), nw = nwords - wfirst;
    for (int c = tid; c < M; c += OCT_T) {
        int o = turn ? M - 1 - c : c, nd = -1;
        if ((S.bm[0][wfirst + (o >> 5)] >> (o & 31)) & 1u) {
            nd = (p1 << 17) | o;
            for (int d = p1 - 1; d >= 0; d--) {
                o = ((n << (2 * (d + 1))) - 1 - o) >> 2;
                if (!((S.bm[1][oct_word0(d, n) + (o >> 5)] >> (o & 31)) & 1u)) nd = (d << 17) | o;
            }
        }
        S.cell[c] = nd;
    }
    __syncthreads();
    for (int i = tid; i < nw; i += OCT_T) S.bm[0][wfirst + i] = 0u;
    __syncthreads();
    for (int c = tid; c < M; c += OCT_T) {
        const int nd = S.cell[c], o = nd & 0x1FFFF;
        if (nd >= 0) atomicOr(&S.bm[0][oct_word0(nd >> 17, n) + (o >> 5)], 1u << (o & 31));
    }
    __syncthreads();
    if (wv == 0) {                               // marks below each word
        int run = 0;
        for (int i0 = 0; i0 < nw; i0 += 64) {
            const int c = i0 + lane < nw ? __popc(S.bm[0][wfirst + i0 + lane]) : 0;
            const int inc = wave_scan(c);
            if (i0 + lane < nw) S.bm[1][wfirst + i0 + lane] = (unsigned)(run + inc - c);
            run += __builtin_amdgcn_readlane(inc, 63);
        }
    }
    __syncthreads();
    for (int c = tid; c < M; c += OCT_T) {
        const int nd = S.cell[c], o = nd & 0x1FFFF;
        if (nd >= 0) {
            const int w = oct_word0(nd >> 17, n) + (o >> 5);
            S.cell[c] = (int)S.bm[1][w] + __popc(S.bm[0][w] & ((1u << (o & 31)) - 1u));
        }
    }
    __syncthreads();
    // each key's node, and (for phase 2) the keys per quadrant of the nodes
    // the last pass made; the bitmaps make way for the counts
    if (tid < size) S.cc[tid] = make_int4(0, 0, 0, 0);
    __syncthreads();
    // quadrant of a key's depth-d cell in its parent: its digit, turned around at even depths
    auto quadrant = [](unsigned place, int d) {
        return (int)((place >> (2 * (OCT_D - d))) & 3u) ^ (d & 1 ? 0 : 3);
    };
#pragma unroll 2
    for (int k = tid; k < K; k += OCT_T) {
        const unsigned place = get(k);
        const int nd = S.cell[place >> sh];
        put(k, place | ((unsigned)nd << 16));
        if (more) atomicAdd((int*)&S.cc[nd] + quadrant(place, p1 + 1), 1);
    }
    __syncthreads();

    // ---- phase 2 (:908-991): split the largest nodes until the quota.  At
    // round r every node of two or more keys has depth p1 + r; every round
    // that does not end the loop grows the list, which holds at most
    // ORB_LIST_CAP nodes.
    for (int depth = p1; more; depth++) {
        // the nodes to expand, keyed by (keys, list position)
        int4 c4 = make_int4(0, 0, 0, 0);
        if (tid < size) c4 = S.cc[tid];
        const int cnt = c4.x + c4.y + c4.z + c4.w;
        if (tid == 0) S.nexp = 0;
        if (tid < ORB_LIST_CAP / 32) S.done[tid] = 0u;
        __syncthreads();
        {
            const unsigned long long b = __ballot(cnt >= 2);
            int base = 0;
            if (lane == 0 && b) base = atomicAdd(&S.nexp, __popcll(b));
            base = __builtin_amdgcn_readfirstlane(base);
            if (cnt >= 2) S.sortk[base + lanes_below(b)] = ((unsigned)cnt << 10) | (unsigned)(ORB_LIST_CAP - 1 - tid);
        }
        __syncthreads();
        const int nE = S.nexp;
        {
            // a key's place in descending order is the number of larger keys;
            // up to 16 lanes share its comparisons
            int lg = 0;
            while (lg < 4 && (nE << (lg + 1)) <= OCT_T) lg++;
            const int i = tid >> lg, step = 1 << lg;
            if (i - (lane >> lg) < nE) {
                const unsigned mine = i < nE ? S.sortk[i] : 0u;
                int rank = 0;
                for (int j = tid & (step - 1); j < nE; j += step) rank += S.sortk[j] > mine ? 1 : 0;
                for (int o = 1; o < step; o <<= 1) rank += __shfl_xor(rank, o, 64);
                if (i < nE && (tid & (step - 1)) == 0)
                    S.order[rank] = (unsigned short)(ORB_LIST_CAP - 1 - (mine & (ORB_LIST_CAP - 1)));
            }
        }
        __syncthreads();
        // gains in processing order, and the first split that reaches the quota
        const int j = tid;
        int nd = 0, nc = 0;
        unsigned occ = 0;
        int4 q4 = make_int4(0, 0, 0, 0);
        if (j < nE) {
            nd = S.order[j];
            q4 = S.cc[nd];
            occ = (q4.x > 0 ? 1u : 0u) | (q4.y > 0 ? 2u : 0u) | (q4.z > 0 ? 4u : 0u) | (q4.w > 0 ? 8u : 0u);
            nc = __popc(occ);
        }
        int all;
        const int ex = block_scan(j < nE ? nc - 1 : 0, S.scan, half, &all);
        const int jstar = min(__syncthreads_count(j < nE && size + ex + nc - 1 < N), nE - 1);
        const bool proc = j <= jstar;
        if (proc) {
            atomicOr(&S.done[nd >> 5], 1u << (nd & 31));
            if (j == jstar) S.cp = ex + nc + j;  // children of the nodes 0 .. jstar
        }
        __syncthreads();
        const int cp = nE > 0 ? S.cp : 0, nsize = cp + size - (jstar + 1);
        if (nsize > ORB_LIST_CAP) return false;  // the general form reports it
        more = nsize < N && nsize != size;
        if (proc) {                              // children in front, the last quadrant first
            S.at[nd] = (unsigned)(cp - (ex + j) - nc) | (occ << 16) | 0x80000000u;
            if (depth + 1 == OCT_D && max(max(q4.x, q4.y), max(q4.z, q4.w)) >= 2) S.deep = 1;
        }
        {
            // kept nodes follow in list order
            const int w = lane < ORB_LIST_CAP / 32 ? (int)S.done[lane] : 0;
            const int below = wave_scan(__popc(w)) - __popc(w);
            const int mw = tid >> 5;
            const int pre = __shfl(below, mw, 64), bits = __shfl(w, mw, 64);
            if (tid < size && !((bits >> (tid & 31)) & 1))
                S.at[tid] = (unsigned)(cp + tid - pre - __popc((unsigned)bits & ((1u << (tid & 31)) - 1u)));
        }
        __syncthreads();
        if (more && S.deep) return false;
        size = nsize;
        if (more) {
            if (tid < size) S.cc[tid] = make_int4(0, 0, 0, 0);
            __syncthreads();
        }
        for (int k = tid; k < K; k += OCT_T) {
            const unsigned v = get(k), place = v & 0xFFFFu, at = S.at[v >> 16];
            const int pos = (int)(at & 0xFFFFu) +
                            (at >> 31 ? __popc(((at >> 16) & 15u) >> (quadrant(place, depth + 1) + 1)) : 0);
            put(k, place | ((unsigned)pos << 16));
            // (past depth OCT_D every node holds one key, and its count alone matters)
            if (more) atomicAdd((int*)&S.cc[pos] + quadrant(place, min(depth + 2, OCT_D)), 1);
        }
        __syncthreads();
    }

    // ---- retain the best response per node; first in key order on ties
    if (tid < size) S.best[tid] = 0ull;
    __syncthreads();
#pragma unroll 4
    for (int k = tid; k < K; k += OCT_T) {
        const unsigned long long kk = gload8u64(L.keys2 + k);
        atomicMax(&S.best[get(k) >> 16], (kk & 0xFFFFFFFF00000000ull) | (0xFFFFFFFFull - (kk & 0xFFFFFFFFull)));
    }
    __syncthreads();
    if (size > min(L.list_cap, ORB_LIST_CAP)) return false;   // the general form reports it
    if (tid < size) {
        const unsigned long long b = S.best[tid];
        gstore8(L.ret + tid, (b & 0xFFFFFFFF00000000ull) | (0xFFFFFFFFull - (b & 0xFFFFFFFFull)));
    }
    if (tid == 0) ctr[ORB_CNT_RET + level] = size;
    return true;
}

// The general form: any candidate set, pass by pass.
__device__ __forceinline__ void octree_general(OctGeneral& S, const LevelJob& L, int level, int* ctr)
{
    const int tid = threadIdx.x, lane = tid & 63;
    // this wavefront's candidate list, and the longest
    const int K0 = min(L.segs[(tid >> 6) * ORB_SEG_STRIDE], L.seg_cap);
    const unsigned long long* list = L.keys + (size_t)(tid >> 6) * L.seg_cap;
    int longest = 0;
    for (int s = 0; s < ORB_SEGS; s++) longest = max(longest, min(L.segs[s * ORB_SEG_STRIDE], L.seg_cap));
    const int N = L.quota;
    const int wC = L.wCell, hC = L.hCell;
    int* node = L.node;
    int total, half = 0;

    // ---- per-cell retry (ORBextractor.cc:1111-1124): a cell keeps its
    // iniThFAST candidates when it has any, else its minThFAST candidates.
    // OCT_REG candidates per thread per round: their keys, then their cell
    // flags, are read together, and one scan places the survivors.  (The
    // candidates' order does not matter: the level kernels append them in
    // no fixed order, and every later step depends only on the set.)
    int K = 0;
    for (int c0 = 0; c0 < longest; c0 += 64 * OCT_REG) {
        unsigned long long key[OCT_REG];
        unsigned char flag[OCT_REG];
#pragma unroll
        for (int m = 0; m < OCT_REG; m++) key[m] = c0 + lane + 64 * m < K0 ? gload8u64(list + c0 + lane + 64 * m) : 0ull;
#pragma unroll
        for (int m = 0; m < OCT_REG; m++) {
            const unsigned ok = (unsigned)key[m];
            flag[m] = gload1(L.cellflag + ((ok >> 20) & 255) * L.nCols + ((ok >> 12) & 255));
        }
        int cnt = 0;
        bool v[OCT_REG];
#pragma unroll
        for (int m = 0; m < OCT_REG; m++) {
            v[m] = c0 + lane + 64 * m < K0 && (key[m] & (flag[m] ? ORB_KEY_INI : ORB_KEY_MIN));
            cnt += v[m] ? 1 : 0;
        }
        int pos = block_scan(cnt, S.scan, half, &total);
#pragma unroll
        for (int m = 0; m < OCT_REG; m++)
            if (v[m]) gstore8(L.keys2 + K + pos++, key[m] & ORB_KEY_RANK);
        K += total;
    }
    __syncthreads();
    const unsigned long long* keys = L.keys2;

    // Each thread keeps the position and list node of its candidates
    // k = tid + OCT_T*m, m < OCT_REG, in registers for every pass; candidates
    // beyond OCT_REG * OCT_T (rare) keep their node in global memory.
    int kx[OCT_REG], ky[OCT_REG], kn[OCT_REG];
    unsigned long long rk[OCT_REG];
#pragma unroll
    for (int m = 0; m < OCT_REG; m++) rk[m] = K > 0 ? gload8u64(keys + min(tid + OCT_T * m, K - 1)) : 0ull;
#pragma unroll
    for (int m = 0; m < OCT_REG; m++) {
        kx[m] = ky[m] = kn[m] = 0;
        if (tid + OCT_T * m < K) key_xy(rk[m], wC, hC, &kx[m], &ky[m]);
    }
    // f(x, y, node&) on every candidate of this thread.
    auto for_keys = [&](auto&& f) {
#pragma unroll
        for (int m = 0; m < OCT_REG; m++)
            if (tid + OCT_T * m < K) f(kx[m], ky[m], kn[m]);
        for (int k = tid + OCT_T * OCT_REG; k < K; k += OCT_T) {
            int x, y;
            key_xy(keys[k], wC, hC, &x, &y);
            int nd = node[k];
            f(x, y, nd);
            node[k] = nd;
        }
    };

    // ---- roots (ORBextractor.cc:695-763)
    if (tid < ORB_MAX_ROOTS) S.cc[tid][0] = 0;
    __syncthreads();
    for_keys([&](int x, int, int& nd) {
        int r = (int)__fdiv_rn((float)x, L.hX);
        r = min(r, L.nIni - 1);
        nd = r;
        atomicAdd(&S.cc[r][0], 1);
    });
    __syncthreads();
    {
        const int c = tid < L.nIni ? S.cc[tid][0] : 0;
        const int pos = block_scan(c > 0 ? 1 : 0, S.scan, half, &total);
        if (tid < L.nIni && c > 0) {
            S.rx[0][pos] = L.root_x[tid] | (L.root_x[tid + 1] << 16);
            S.ry[0][pos] = 0 | ((L.maxBorderY - ORB_MIN_BORDER) << 16);
            S.cnt[0][pos] = c;
            S.seq[0][pos] = tid;
        }
        if (tid < L.nIni) S.keep[tid] = (short)pos;
    }
    __syncthreads();
    for_keys([&](int, int, int& nd) { nd = S.keep[nd]; });
    int cur = 0;
    int size = total;
    bool phase2 = false;
    __syncthreads();

    // ---- phase 1: full passes (ORBextractor.cc:779-893).  Every pass
    // that does not end the loop grows the list, which holds at most
    // ORB_LIST_CAP nodes, so a pass count beyond that is an internal error.
    for (int pass = 0;; pass++) {
        if (pass > ORB_LIST_CAP) {
            if (tid == 0) atomicOr(&ctr[ORB_CNT_ERR], ORB_ERR_LIST);
            size = 0;
            break;
        }
        const int prev = size;
        for (int i = tid; i < size; i += OCT_T) S.cc[i][0] = S.cc[i][1] = S.cc[i][2] = S.cc[i][3] = 0;
        __syncthreads();
        for_keys([&](int x, int y, int& nd) {
            const int i = nd;
            if (S.cnt[cur][i] >= 2) atomicAdd(&S.cc[i][quad_of(S.rx[cur][i], S.ry[cur][i], x, y)], 1);
        });
        __syncthreads();
        const int i = tid;
        const bool split = i < size && S.cnt[cur][i] >= 2;
        int nc = 0;
        if (split) nc = (S.cc[i][0] > 0) + (S.cc[i][1] > 0) + (S.cc[i][2] > 0) + (S.cc[i][3] > 0);
        const int kp = (i < size && !split) ? 1 : 0;
        int C, nkeep;
        const int ex_nc = block_scan(nc, S.scan, half, &C);
        const int ex_kp = block_scan(kp, S.scan, half, &nkeep);
        const int nsize = C + nkeep;
        int nexp = 0;
        if (nsize <= ORB_LIST_CAP) {
            const int nb = cur ^ 1;
            if (split) {
                const int base = C - ex_nc - nc;
                int r = 0;
                for (int q = 3; q >= 0; q--) {
                    const int c = S.cc[i][q];
                    if (c > 0) {
                        const int pos = base + r++;
                        int crx, cry;
                        child_rect(S.rx[cur][i], S.ry[cur][i], q, &crx, &cry);
                        S.rx[nb][pos] = crx;
                        S.ry[nb][pos] = cry;
                        S.cnt[nb][pos] = c;
                        S.seq[nb][pos] = ex_nc + (nc - r);   // creation order n1..n4
                        S.map[i][q] = (short)pos;
                        nexp += c >= 2;
                    } else {
                        S.map[i][q] = -1;
                    }
                }
            } else if (kp) {
                const int pos = C + ex_kp;
                S.rx[nb][pos] = S.rx[cur][i];
                S.ry[nb][pos] = S.ry[cur][i];
                S.cnt[nb][pos] = S.cnt[cur][i];
                S.seq[nb][pos] = S.seq[cur][i];
                S.keep[i] = (short)pos;
            }
        }
        int nToExpand;
        block_scan(nexp, S.scan, half, &nToExpand);
        if (nsize > ORB_LIST_CAP) {
            if (tid == 0) atomicOr(&ctr[ORB_CNT_ERR], ORB_ERR_LIST);
            size = 0;
            break;
        }
        for_keys([&](int x, int y, int& nd) {
            const int n0 = nd;
            nd = S.cnt[cur][n0] >= 2 ? S.map[n0][quad_of(S.rx[cur][n0], S.ry[cur][n0], x, y)] : S.keep[n0];
        });
        cur ^= 1;
        size = nsize;
        __syncthreads();
        if (size >= N || size == prev) break;
        if (size + nToExpand * 3 > N) {
            phase2 = true;
            break;
        }
    }

    // ---- phase 2: split the largest nodes until the quota (:908-991); as
    // in phase 1, every round that does not end the loop grows the list.
    for (int round = 0; phase2; round++) {
        if (round > ORB_LIST_CAP) {
            if (tid == 0) atomicOr(&ctr[ORB_CNT_ERR], ORB_ERR_LIST);
            size = 0;
            break;
        }
        const int prev = size;
        for (int i = tid; i < size; i += OCT_T) S.cc[i][0] = S.cc[i][1] = S.cc[i][2] = S.cc[i][3] = 0;
        __syncthreads();
        for_keys([&](int x, int y, int& nd) {
            const int i = nd;
            if (S.cnt[cur][i] >= 2) atomicAdd(&S.cc[i][quad_of(S.rx[cur][i], S.ry[cur][i], x, y)], 1);
        });
        // Expandable nodes, sorted by (size, creation order), largest first.
        const bool e = tid < size && S.cnt[cur][tid] >= 2;
        int nE;
        const int ex_e = block_scan(e ? 1 : 0, S.scan, half, &nE);
        // The keys are distinct (they carry the node index), so a key's
        // place in descending order is the number of larger keys.  S.keep
        // holds each node's place (32767: not expandable).
        if (e)
            S.sortk[ex_e] = ((unsigned long long)S.cnt[cur][tid] << 32) |
                            ((unsigned long long)(unsigned)S.seq[cur][tid] << 16) | (unsigned)tid;
        if (tid < size) S.keep[tid] = 32767;
        __syncthreads();
        {
            // up to 16 lanes share a key's comparisons
            int lg = 0;
            while (lg < 4 && (nE << (lg + 1)) <= OCT_T) lg++;
            const int i = tid >> lg, step = 1 << lg;
            const bool mine_ok = i < nE;
            const unsigned long long mine = S.sortk[mine_ok ? i : 0];
            int rank = 0;
            for (int j2 = tid & (step - 1); j2 < nE; j2 += step) rank += S.sortk[j2] > mine;
            for (int o2 = 1; o2 < step; o2 <<= 1) rank += __shfl_xor(rank, o2, 64);
            if (mine_ok && (tid & (step - 1)) == 0) {
                S.best[rank] = mine;             // S.best is free until the retain step
                S.keep[mine & 0xFFFF] = (short)rank;
            }
        }
        __syncthreads();
        // Gains in processing order and the first split reaching the quota.
        const int j = tid;
        int node_j = -1, nc = 0;
        if (j < nE) {
            node_j = (int)(S.best[j] & 0xFFFF);
            nc = (S.cc[node_j][0] > 0) + (S.cc[node_j][1] > 0) + (S.cc[node_j][2] > 0) + (S.cc[node_j][3] > 0);
        }
        int gsum;
        const int ex_g = block_scan(j < nE ? nc - 1 : 0, S.scan, half, &gsum);
        if (tid == 0) S.vars[0] = nE - 1;
        __syncthreads();
        if (j < nE && size + ex_g + nc - 1 >= N) atomicMin(&S.vars[0], j);
        __syncthreads();
        const int jstar = S.vars[0];
        const bool proc = j <= jstar && j < nE;
        // Kept list nodes: all but the processed ones (place <= jstar).  One
        // scan for the processed nodes' children (<= 4 * ORB_LIST_CAP < 2^16)
        // and the kept nodes (<= ORB_LIST_CAP).
        static_assert(4 * ORB_LIST_CAP < (1 << 16) && ORB_LIST_CAP <= OCT_T, "octree list packing");
        const bool kp = tid < size && S.keep[tid] > jstar;
        int tot;
        const int ex = block_scan((proc ? nc : 0) | ((kp ? 1 : 0) << 16), S.scan, half, &tot);
        const int ex_nc = ex & 0xFFFF, ex_kp = ex >> 16, Cp = tot & 0xFFFF, nkeep = tot >> 16;
        const int nsize = Cp + nkeep;
        if (nsize > ORB_LIST_CAP) {
            if (tid == 0) atomicOr(&ctr[ORB_CNT_ERR], ORB_ERR_LIST);
            size = 0;
            break;
        }
        const int nb = cur ^ 1;
        if (proc) {
            const int i = node_j;
            const int base = Cp - ex_nc - nc;
            int r = 0;
            for (int q = 3; q >= 0; q--) {
                const int c = S.cc[i][q];
                if (c > 0) {
                    const int pos = base + r++;
                    int crx, cry;
                    child_rect(S.rx[cur][i], S.ry[cur][i], q, &crx, &cry);
                    S.rx[nb][pos] = crx;
                    S.ry[nb][pos] = cry;
                    S.cnt[nb][pos] = c;
                    S.seq[nb][pos] = ex_nc + (nc - r);
                    S.map[i][q] = (short)pos;
                } else {
                    S.map[i][q] = -1;
                }
            }
        }
        int keeppos = -1;
        if (kp) {
            const int i = tid;
            keeppos = Cp + ex_kp;
            S.rx[nb][keeppos] = S.rx[cur][i];
            S.ry[nb][keeppos] = S.ry[cur][i];
            S.cnt[nb][keeppos] = S.cnt[cur][i];
            S.seq[nb][keeppos] = S.seq[cur][i];
        }
        __syncthreads();
        if (tid < size) S.keep[tid] = (short)(kp ? keeppos : -1);
        __syncthreads();
        for_keys([&](int x, int y, int& nd) {
            const int n0 = nd;
            const int kv = S.keep[n0];
            nd = kv < 0 ? S.map[n0][quad_of(S.rx[cur][n0], S.ry[cur][n0], x, y)] : kv;
        });
        cur ^= 1;
        size = nsize;
        __syncthreads();
        if (size >= N || size == prev) break;
    }

    // ---- retain the best response per node; first in key order on ties
    for (int i = tid; i < size; i += OCT_T) S.best[i] = 0ull;
    __syncthreads();
    auto retain = [&](unsigned long long key, int nd) {
        const unsigned long long packed = (key & 0xFFFFFFFF00000000ull) | (0xFFFFFFFFull - (key & 0xFFFFFFFFull));
        atomicMax(&S.best[nd], packed);
    };
#pragma unroll
    for (int m = 0; m < OCT_REG; m++)
        if (tid + OCT_T * m < K) retain(gload8u64(keys + tid + OCT_T * m), kn[m]);
    for (int k = tid + OCT_T * OCT_REG; k < K; k += OCT_T) retain(keys[k], node[k]);
    __syncthreads();
    const int cap = min(L.list_cap, ORB_LIST_CAP);
    if (size > cap) {
        if (tid == 0) atomicOr(&ctr[ORB_CNT_ERR], ORB_ERR_LIST);
        size = 0;
    }
    for (int i = tid; i < size; i += OCT_T) {
        const unsigned long long p = S.best[i];
        gstore8(L.ret + i, (p & 0xFFFFFFFF00000000ull) | (0xFFFFFFFFull - (p & 0xFFFFFFFFull)));
    }
    if (tid == 0) ctr[ORB_CNT_RET + level] = size;
}

__global__ __launch_bounds__(OCT_T, 8) void octree_kernel(const ImageJob* __restrict__ jobs, int max_levels)
{
    __shared__ union {
        OctFast f;
        OctGeneral g;
    } S;
    const int jb = blockIdx.x / max_levels, level = blockIdx.x % max_levels;
    const ImageJob& J = jobs[jb];
    if (level >= J.nlevels) return;
    const LevelJob& L = J.lv[level];
    if (octree_fast(S.f, L, level, J.counters)) return;
    __syncthreads();
    octree_general(S.g, L, level, J.counters);
}

// ============================================================== describe
// fastAtan2 (OpenCV 2.4/3.x): degree-7 odd polynomial, degrees in [0,360).
__device__ __forceinline__ float fast_atan2_dev(float y, float x)
{
    const float P1 = 0.9997878412794807f * (float)(180 / 3.1415926535897932384626433832795);
    const float P3 = -0.3258083974640975f * (float)(180 / 3.1415926535897932384626433832795);
    const float P5 = 0.1555786518463281f * (float)(180 / 3.1415926535897932384626433832795);
    const float P7 = -0.04432655554792128f * (float)(180 / 3.1415926535897932384626433832795);
    const float ax = fabsf(x), ay = fabsf(y);
    float a, c, c2;
    if (ax >= ay) {
        c = __fdiv_rn(ay, ax + (float)DBL_EPSILON);
        c2 = c * c;
        a = (((P7 * c2 + P5) * c2 + P3) * c2 + P1) * c;
    } else {
        c = __fdiv_rn(ax, ay + (float)DBL_EPSILON);
        c2 = c * c;
        a = 90.f - (((P7 * c2 + P5) * c2 + P3) * c2 + P1) * c;
    }
    if (x < 0) a = 180.f - a;
    if (y < 0) a = 360.f - a;
    return a;
}

// cos/sin of a float angle, evaluated in double by Cody-Waite reduction and
// Taylor series, then rounded to float: a fixed method so that the CPU
// statement and this kernel agree bit for bit.
__device__ __forceinline__ void sincos_canonical_dev(double x, double* s, double* c)
{
    const double kPio2Hi = 1.57079632673412561417e+00;
    const double kPio2Lo = 6.07710050650619224932e-11;
    const double kTwoOverPi = 6.36619772367581382433e-01;
    const double kd = rint(x * kTwoOverPi);
    const int k = (int)kd;
    const double r = (x - kd * kPio2Hi) - kd * kPio2Lo;
    const double r2 = r * r;
    double ps = 1.0 / 355687428096000.0;
    ps = ps * r2 - 1.0 / 1307674368000.0;
    ps = ps * r2 + 1.0 / 6227020800.0;
    ps = ps * r2 - 1.0 / 39916800.0;
    ps = ps * r2 + 1.0 / 362880.0;
    ps = ps * r2 - 1.0 / 5040.0;
    ps = ps * r2 + 1.0 / 120.0;
    ps = ps * r2 - 1.0 / 6.0;
    const double sr = r + r * r2 * ps;
    double pc = 1.0 / 6402373705728000.0;
    pc = pc * r2 - 1.0 / 20922789888000.0;
    pc = pc * r2 + 1.0 / 87178291200.0;
    pc = pc * r2 - 1.0 / 479001600.0;
    pc = pc * r2 + 1.0 / 3628800.0;
    pc = pc * r2 - 1.0 / 40320.0;
    pc = pc * r2 + 1.0 / 720.0;
    pc = pc * r2 - 1.0 / 24.0;
    pc = pc * r2 + 0.5;
    const double cr = 1.0 - r2 * pc;
    switch (k & 3) {
    case 0: *s = sr; *c = cr; break;
    case 1: *s = cr; *c = -sr; break;
    case 2: *s = -sr; *c = -cr; break;
    default: *s = -cr; *c = sr; break;
    }
}

// A 16-lane group per kept keypoint, four per wavefront; a workgroup serves
// 16 keypoints of one (image, level), so the level's geometry and output
// offset are uniform across it.  The lanes of a group share the rows of its
// patches; lane j takes BRIEF pairs 16j .. 16j+15 (descriptor bytes 2j, 2j+1).
// Bound: latency of the patch reads (185 MB from memory in a batch of 128 images
// of 1241 x 376), with 5 wavefronts a SIMD and half the vector issue slots used.
#define DESC_G 16
static_assert(256 / DESC_G == ORB_DESC_KPB, "describe blocks are counted on the host");
__global__ __launch_bounds__(256) void describe_kernel(const ImageJob* __restrict__ jobs,
                                                       const RunTable* __restrict__ rt)
{
    __shared__ uint2 s_brief[ORB_DESC_KPB][37 * 5];   // per group: 37 rows x 40 bytes
    __shared__ uint4 s_pat[64];
    __shared__ uint4 s_mask[4 * 16 * 3];
    const int sub = threadIdx.x & (DESC_G - 1), grp = threadIdx.x / DESC_G;
    const int nseg = rt->njobs * rt->max_levels;
    const int blk = xcd_block(blockIdx.x, gridDim.x);
    const int dpj = rt->desc_per_job;
    const int f = dpj > 0 ? (blk / dpj) * rt->max_levels +
                                find_segment(rt->desc_start + (blk / dpj) * rt->max_levels, rt->max_levels, blk)
                          : find_segment(rt->desc_start, nseg, blk);
    const int jb = f / rt->max_levels, level = f % rt->max_levels;
    const ImageJob& J = jobs[jb];
    const int* ctr = J.counters;
    int base = 0, total = 0;
    for (int l = 0; l < J.nlevels; l++) {
        const int c = (int)gload4((const uint8_t*)(ctr + ORB_CNT_RET + l));
        base += l < level ? c : 0;
        total += c;
    }
    const int idx = (blk - rt->desc_start[f]) * ORB_DESC_KPB + grp;
    if (level == 0 && idx == 0 && sub == 0) J.counters[ORB_CNT_NOUT] = total;
    // The 256 BRIEF pairs (one dword of 4 signed bytes each) into LDS, laid
    // out so that lane j's k-th 16-byte read holds its pairs 16j+4k .. +3
    // and the 16 lanes of a group read consecutive 16-byte words.
    {
        const int t = threadIdx.x;
        ((unsigned*)s_pat)[(((t >> 2) & 3) * 16 + (t >> 4)) * 4 + (t & 3)] = ((const unsigned*)c_pattern)[t];
        if (t < 4 * 16 * 3) s_mask[t] = c_icmask[t];
    }
    __syncthreads();
    if (level >= J.nlevels || idx >= (int)gload4((const uint8_t*)(ctr + ORB_CNT_RET + level))) return;   // the whole group leaves
    const LevelJob& L = J.lv[level];
    const unsigned long long key = gload8u64(L.ret + idx);
    int xr, yr;
    key_xy(key, L.wCell, L.hCell, &xr, &yr);
    const int cx = xr + ORB_MIN_BORDER, cy = yr + ORB_MIN_BORDER;
    const int pitch = L.pitch;

    // Both patches are read with dword-aligned loads issued together, before
    // any use: the 31x31 orientation patch of the level and the 37x37 window
    // of the blurred level that every rotated BRIEF sample falls in (pattern
    // radius <= 18.39 px).  Keypoints lie >= 19 px inside the level (x <= w-20,
    // y <= h-20), so the pieces end at most 13 (level) and 2 (blur) bytes past
    // a row's last pixel, and every row read has successors: inside the level's
    // buffer.
    const int xa0 = (cx - 15) & ~3;               // 31 px + <= 3 of alignment: 9 dwords a row
    const int xb0 = (cx - 18) & ~3;               // 37 px + <= 3 of alignment: 10 dwords a row
    // Neighbouring lanes read neighbouring pieces of a row, so that a load meets
    // 64 / 3 or 64 / 5 rows' cache lines and not 64: the orientation patch in 93
    // pieces of 16 bytes (3 a row, the last of one dword in use), the blur window
    // in 185 of 8 bytes (5 a row), which is also its layout in LDS.  (A lane per
    // row was 68 M cache accesses on 128 images of 1241 x 376, this is 39 M: 169
    // us and 154; 64 images of four sizes 46 and 44.)
    uint4 pa[6];
    uint2 pb[12];
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const int i = min(sub + 16 * k, 92), r = (i * 171) >> 9;          // i / 3
        pa[k] = gload16(L.lvl + (unsigned)((cy - 15 + r) * pitch + xa0 + 16 * (i - 3 * r)));
    }
#pragma unroll
    for (int k = 0; k < 12; k++) {
        const int i = min(sub + 16 * k, 184), r = (i * 205) >> 10;        // i / 5
        pb[k] = gload8(L.blur + (unsigned)((cy - 18 + r) * pitch + xb0 + 8 * (i - 5 * r)));
    }

    // IC_Angle (ORBextractor.cc:94-141): m10 = sum u*I, m01 = sum v*I over
    // the disc |u| <= umax[|v|].  Per dword of 4 pixels: the disc's byte mask
    // (a table over the row's |v| and the patch's alignment), then
    // v_dot4_u32_u8 for the masked sum and for sum (u+20)*I.
    const int al = (cx - 15) & 3;                 // u of byte k of dword c: 4c + k - 15 - al
    const unsigned w0 = (unsigned)(5 - al) * 0x01010101u + 0x03020100u;   // bytes u+20 of dword 0
    int m01 = 0;
    unsigned s1 = 0, su = 0;
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const int i = min(sub + 16 * k, 92), r = (i * 171) >> 9, c = i - 3 * r, v = r - 15;
        uint4 d = pa[k];
        const uint4 m = s_mask[(al * 16 + max(v, -v)) * 3 + c];
        d.x &= m.x, d.y &= m.y, d.z &= m.z, d.w &= m.w;
        unsigned row = __builtin_amdgcn_udot4(d.x, 0x01010101u, 0u, false);
        row = __builtin_amdgcn_udot4(d.y, 0x01010101u, row, false);
        row = __builtin_amdgcn_udot4(d.z, 0x01010101u, row, false);
        row = __builtin_amdgcn_udot4(d.w, 0x01010101u, row, false);
        const unsigned w = w0 + __builtin_amdgcn_perm(0u, (unsigned)(16 * c), 0u);   // 16 c in each byte
        unsigned us = __builtin_amdgcn_udot4(d.x, w, 0u, false);
        us = __builtin_amdgcn_udot4(d.y, w + 0x04040404u, us, false);
        us = __builtin_amdgcn_udot4(d.z, w + 0x08080808u, us, false);
        us = __builtin_amdgcn_udot4(d.w, w + 0x0C0C0C0Cu, us, false);
        if (k < 5 || sub < 13) {                  // 93 pieces
            m01 += v * (int)row;
            s1 += row;
            su += us;
        }
    }
    int m10 = (int)su - 20 * (int)s1;
    m10 = (int)row16_sum((unsigned)m10);
    m01 = (int)row16_sum((unsigned)m01);
    const float angle_deg = fast_atan2_dev((float)m01, (float)m10);

    const float factorPI = (float)(3.1415926535897932384626433832795 / 180.f);
    const float angle = angle_deg * factorPI;
    double sd, cd;
    sincos_canonical_dev((double)angle, &sd, &cd);
    const float a = (float)cd, b = (float)sd;

    // The blur window goes to LDS only now, so that its reads stay in flight
    // under the orientation and rotation arithmetic above.
    uint2* win = s_brief[grp];
#pragma unroll
    for (int k = 0; k < 12; k++)
        if (k < 11 || sub < 9) win[sub + 16 * k] = pb[k];     // 185 pieces

    // Rotated BRIEF (ORBextractor.cc:153-204) on the blurred level, sampled
    // from the staged window (row stride 40 bytes, centre at row 18).
    // cvRound of a sample coordinate t (|t| < 19) is read from the bits of
    // t + 1.5 * 2^23, whose low 23 bits hold 2^22 + rint(t): the sum rounds
    // to the nearest integer, ties to even, as rint does.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float kRound = 12582912.0f;
    // sample (iy, ix) is byte (18 + iy) * 40 + (cx - xb0) + ix of the window;
    // with both read as 2^22 + i in the low 24 bits, the byte is
    // (2^22 + iy) * 40 + (bits of x) - kBias
    const unsigned kBias = (1u << 22) * 40u + 0x4B400000u - 18u * 40u - (unsigned)(cx - xb0);
    const uint8_t* wb = (const uint8_t*)win;
    unsigned bits = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const uint4 q = s_pat[k * 16 + sub];
        const unsigned qd[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int d = (int)qd[e];
            const float px0 = (float)(signed char)d, py0 = (float)(signed char)(d >> 8);
            const float px1 = (float)(signed char)(d >> 16), py1 = (float)(d >> 24);
            const float y0r = px0 * b + py0 * a, x0r = px0 * a - py0 * b;
            const float y1r = px1 * b + py1 * a, x1r = px1 * a - py1 * b;
            const unsigned o0 = (__float_as_uint(y0r + kRound) & 0xFFFFFFu) * 40u + __float_as_uint(x0r + kRound) - kBias;
            const unsigned o1 = (__float_as_uint(y1r + kRound) & 0xFFFFFFu) * 40u + __float_as_uint(x1r + kRound) - kBias;
            const int i0 = wb[o0], i1 = wb[o1];
            bits |= (unsigned)(i0 < i1) << (4 * k + e);
        }
    }
    const int out = base + idx;
    gstore2(J.desc + (size_t)out * 32 + 2 * sub, (unsigned short)bits);
    if (sub == 0) {
        const float sc = L.scale;
        OrbKeyPoint kp;
        float fx = (float)cx, fy = (float)cy;
        if (level != 0) {
            fx = fx * sc;
            fy = fy * sc;
        }
        kp.x = fx;
        kp.y = fy;
        kp.size = (float)(int)(31 * sc);
        kp.angle = angle_deg;
        kp.response = (float)(unsigned)(key >> 32);
        kp.octave = level;
        kp.class_id = -1;
        uint8_t* kd = (uint8_t*)(J.kps + out);     // 28 bytes: 16 + 8 + 4
        gstore16(kd, make_uint4(__float_as_uint(kp.x), __float_as_uint(kp.y), __float_as_uint(kp.size),
                                __float_as_uint(kp.angle)));
        *(__attribute__((address_space(1))) orb_v2u*)(kd + 16) =
            orb_v2u{__float_as_uint(kp.response), (unsigned)kp.octave};
        gstore4(kd + 24, (unsigned)kp.class_id);
    }
}

// ============================================================ zero fill
// Counters and per-cell flags of every job (one workgroup per job), for runs
// whose pyramid launch does not clear them.
__global__ void zero_counters_kernel(const ImageJob* __restrict__ jobs, int njobs)
{
    if ((int)blockIdx.x < njobs) zero_job(jobs[blockIdx.x]);
}

// ========================================================= Hamming helpers
__device__ __forceinline__ int hamming32(const uint4 a0, const uint4 a1, const uint8_t* b)
{
    const uint4 b0 = *(const uint4*)b, b1 = *(const uint4*)(b + 16);
    return __popc(a0.x ^ b0.x) + __popc(a0.y ^ b0.y) + __popc(a0.z ^ b0.z) + __popc(a0.w ^ b0.w) +
           __popc(a1.x ^ b1.x) + __popc(a1.y ^ b1.y) + __popc(a1.z ^ b1.z) + __popc(a1.w ^ b1.w);
}

// ================================================================ stereo
// Frame::ComputeStereoMatches (Frame.cc:831-1082), a 16-lane group per left
// keypoint.  Search: right keypoints whose row band [floor(y-2s), ceil(y+2s)]
// holds row (size_t)vL, octave within +-1, uR in [uL-maxD, uL]; best is the
// smallest (distance, index) below TH_HIGH.  Refinement: 11x11 SAD of
// centre-subtracted patches over 11 shifts, parabola fit, depth = bf/disp.

// Group each pair's right keypoints by (octave, level-0 row bucket)
// (counting sort in LDS, one workgroup per pair) and lay them out in that
// order as 16-byte records {minr, maxr, index << 4 | octave, x} (the row band
// of Frame.cc:867-882, with the same float statements) and 32-byte
// descriptors; plus, per octave and level-0 row, the entry range of that
// octave's buckets that can hold the row in a band.  Order inside a bucket is free: the search keeps the smallest
// (distance, index), which does not depend on the visiting order.
#define STEREO_NB 4096               // buckets: rows >> qs
#define STEREO_T 1024
#define STEREO_PER_T 4               // right keypoints per thread (<= 4096)
__global__ __launch_bounds__(STEREO_T) void stereo_prep_kernel(const StereoArgs* __restrict__ args)
{
    __shared__ int s_cnt[STEREO_NB + 1];
    __shared__ int s_part[STEREO_T / 64];
    const StereoArgs& A = args[blockIdx.x];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int n = min(min(*A.nr, A.cap_r), STEREO_T * STEREO_PER_T);
    const int nrows = A.nrows, nlev = A.nlev;
    int qs = 0;
    while (nlev * (((nrows - 1) >> qs) + 1) > STEREO_NB) qs++;
    const int nb = ((nrows - 1) >> qs) + 1;      // row buckets per octave
    const int nk = nlev * nb;                    // keys: octave * nb + row bucket
    // Bucket of a y: floor(y) clamped to the rows (NaN to row 0), >> qs.
    auto bucket = [nrows, qs](float y) {
        const float f = floorf(y);
        const int r = !(f > 0.f) ? 0 : (f >= (float)(nrows - 1) ? nrows - 1 : (int)f);
        return r >> qs;
    };
    for (int j = t; j <= nk; j += STEREO_T) s_cnt[j] = 0;
    __syncthreads();
    // Each thread's keypoints and descriptors are read once, here; the
    // scatter after the scan uses the registers.
    int eb[STEREO_PER_T], er[STEREO_PER_T], ko[STEREO_PER_T];
    uint2 kxy[STEREO_PER_T];
    uint4 kd0[STEREO_PER_T], kd1[STEREO_PER_T];
#pragma unroll
    for (int k = 0; k < STEREO_PER_T; k++) {
        const int i = t + STEREO_T * k;
        eb[k] = 0;
        ko[k] = 0;
        kxy[k] = make_uint2(0u, 0u);
        kd0[k] = kd1[k] = make_uint4(0u, 0u, 0u, 0u);
        if (i < n) {
            const uint8_t* kb = (const uint8_t*)(A.kr + i);
            kxy[k] = gload8(kb + offsetof(OrbKeyPoint, x));
            ko[k] = (int)gload4(kb + offsetof(OrbKeyPoint, octave));
            const uint8_t* d = A.dr + (size_t)i * 32;
            kd0[k] = gload16(d);
            kd1[k] = gload16(d + 16);
            eb[k] = min(ko[k], nlev - 1) * nb + bucket(__uint_as_float(kxy[k].y));
        }
        er[k] = i < n ? atomicAdd(&s_cnt[eb[k]], 1) : 0;
    }
    __syncthreads();
    // Exclusive scan of the nk counts: 4 per thread, wavefront scans, then
    // the 16 wavefront totals.
    int loc[4], sum = 0;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int j = 4 * t + k;
        loc[k] = sum;
        sum += j < nk ? s_cnt[j] : 0;
    }
    int inc = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
    }
    if (lane == 63) s_part[wv] = inc;
    __syncthreads();
    int base = inc - sum;
    for (int k = 0; k < wv; k++) base += s_part[k];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int j = 4 * t + k;
        if (j < nk) s_cnt[j] = base + loc[k];
    }
    if (t == 0) s_cnt[nk] = n;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < STEREO_PER_T; k++) {
        const int i = t + STEREO_T * k;
        if (i < n) {
            const uint2 xy = kxy[k];
            const int oct = ko[k];
            const float ky = __uint_as_float(xy.y);
            const float r = 2.0f * A.scale[oct];
            const int maxr = (int)ceilf(ky + r);
            const int minr = (int)floorf(ky - r);
            const int pos = s_cnt[eb[k]] + er[k];
            gstore16((uint8_t*)(A.srec + pos), make_uint4((unsigned)minr, (unsigned)maxr, (unsigned)((i << 4) | oct), xy.x));
            uint8_t* o = A.sdesc + (size_t)pos * 32;
            gstore16(o, kd0[k]);
            gstore16(o + 16, kd1[k]);
        }
    }
    // A candidate of octave o for row `row` has y in (row - 1 - r, row + 1 + r),
    // r = 2 * scale[o]; one more row each side absorbs the rounding of these
    // bounds.  rows[o * nrows + row]: the entries of those buckets of octave o.
    for (int idx = t; idx < nlev * nrows; idx += STEREO_T) {
        const int o = idx / nrows, row = idx - o * nrows;
        const float r = 2.0f * A.scale[o];
        const int blo = bucket((float)row - 2.0f - r), bhi = bucket((float)row + 2.0f + r);
        *(__attribute__((address_space(1))) orb_v2u*)(A.rows + idx) =
            orb_v2u{(unsigned)s_cnt[o * nb + blo], (unsigned)s_cnt[o * nb + bhi + 1]};
    }
}

// One 32-bit load of a patch row, bytewise where it would pass the level's
// right edge.
__device__ __forceinline__ unsigned patch_dword(const uint8_t* rp, int x, int w)
{
    if (x + 3 < w) return *(const unsigned*)(rp + x);
    unsigned d = 0;
    for (int b = 0; b < 4; b++)
        if (x + b < w) d |= (unsigned)rp[x + b] << (8 * b);
    return d;
}


// grid (ceil(max left capacity / 16), pairs): lanes 16g .. 16g+15 of a
// wavefront serve one left keypoint.  Every branch is uniform within a
// group, and cross-lane steps stay inside it.
//   search: the group's lanes stride over the row's candidate range;
//   refinement: lane r < 11 holds patch row r of both images in registers
//   as 16-bit pairs and accumulates its row's part of the 11 shift SADs with
//   v_sad_u16 (two absolute differences per instruction), as
//   |(l - cL) - (r - cR)| = |(l + cR - cL + 256) - (r + 256)|, both sides in
//   [0, 766]; the row parts are summed across the group with DPP, two shifts
//   per dword (a total is at most 121 * 510 < 2^16).
#define ST_G 16
#ifndef ST_CHUNK
#define ST_CHUNK 2
#endif
__global__ __launch_bounds__(256) void stereo_kernel(const StereoArgs* __restrict__ args)
{
    const int sub = threadIdx.x & (ST_G - 1);
    const int gbase = threadIdx.x & 63 & ~(ST_G - 1);
    // XCD-aware order: each XCD takes a contiguous run of (pair, keypoint
    // block), so the patch rows that a pair's neighbouring keypoints share
    // are fetched into one L2 rather than into all of them.
    const int lb = xcd_block(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    const int pair = lb / gridDim.x, kblk = lb - pair * gridDim.x;
    const StereoArgs& A = args[pair];
    const int iL = kblk * (256 / ST_G) + (int)(threadIdx.x / ST_G);
    const int nl = *A.nl, nr = *A.nr;
    if (iL >= nl || iL >= A.cap_l) return;             // the whole group leaves
    float outU = -1.0f, outD = -1.0f;
    int outSad = -1;
    const uint8_t* kpb = (const uint8_t*)(A.kl + iL);
    const uint2 kxy = gload8(kpb + offsetof(OrbKeyPoint, x));
    const uint4 a0 = gload16(A.dl + (unsigned)iL * 32u), a1 = gload16(A.dl + (unsigned)iL * 32u + 16u);
    const int levelL = (int)gload4(kpb + offsetof(OrbKeyPoint, octave));
    const float vL = __uint_as_float(kxy.y), uL = __uint_as_float(kxy.x);
    const int row = (int)vL;
    const float minZ = A.mb;
    const float minD = 0;
    const float maxD = A.bf / minZ;
    const float minU = uL - maxD;
    const float maxU = uL - minD;
    bool go = row >= 0 && row < A.nrows && !(maxU < 0);
    // The level both patches are read from (octaves are validated on entry
    // and produced in range by the extractor).
    const LevelJob& LL = A.left->lv[levelL];
    const LevelJob& LR = A.right->lv[levelL];
    const uint8_t* pl = LL.lvl;
    const uint8_t* pr = LR.lvl;
    const int pitchL = LL.pitch, pitchR = LR.pitch, wL = LL.w, hL = LL.h, wR = LR.w, hR = LR.h;
    int bestDist = 100, bestIdx = INT_MAX;
    float bestU = 0.f;
    if (go) {
        (void)nr;
        // Octaves levelL-1 .. levelL+1 only (Frame.cc:929), each over the
        // entries of its own row band.
        for (int oc = max(levelL - 1, 0); oc <= min(levelL + 1, A.nlev - 1); oc++) {
            const int2 rg = A.rows[oc * A.nrows + row];
            // Chunks of ST_CHUNK candidates per lane: the records are loaded
            // together, then the descriptors of those that pass the band, octave
            // and uR tests, so each chunk waits on memory twice.
            for (int c0 = rg.x + sub; c0 < rg.y; c0 += ST_CHUNK * ST_G) {
                int4 rec[ST_CHUNK];
#pragma unroll
                for (int u = 0; u < ST_CHUNK; u++) {
                    const int c = c0 + u * ST_G;
                    if (c < rg.y) {
                        const uint4 q = gload16((const uint8_t*)A.srec + (unsigned)c * 16u);
                        rec[u] = make_int4((int)q.x, (int)q.y, (int)q.z, (int)q.w);
                    } else {
                        rec[u] = make_int4(1, 0, 0, 0);   // minr > maxr: never a candidate
                    }
                }
                bool pass[ST_CHUNK];
#pragma unroll
                for (int u = 0; u < ST_CHUNK; u++) {
                    const int oct = rec[u].z & 15;
                    const float uR = __int_as_float(rec[u].w);
                    pass[u] = row >= rec[u].x && row <= rec[u].y && oct >= levelL - 1 && oct <= levelL + 1 &&
                              uR >= minU && uR <= maxU;
                }
                uint4 b0[ST_CHUNK], b1[ST_CHUNK];
#pragma unroll
                for (int u = 0; u < ST_CHUNK; u++) {
                    if (pass[u]) {
                        const uint8_t* d = A.sdesc + (unsigned)(c0 + u * ST_G) * 32u;
                        b0[u] = gload16(d);
                        b1[u] = gload16(d + 16);
                    }
                }
#pragma unroll
                for (int u = 0; u < ST_CHUNK; u++) {
                    if (pass[u]) {
                        const int iR = rec[u].z >> 4;
                        const int dist = __popc(a0.x ^ b0[u].x) + __popc(a0.y ^ b0[u].y) + __popc(a0.z ^ b0[u].z) +
                                         __popc(a0.w ^ b0[u].w) + __popc(a1.x ^ b1[u].x) + __popc(a1.y ^ b1[u].y) +
                                         __popc(a1.z ^ b1[u].z) + __popc(a1.w ^ b1[u].w);
                        if (dist < bestDist || (dist == bestDist && iR < bestIdx)) {
                            bestDist = dist;
                            bestIdx = iR;
                            bestU = __int_as_float(rec[u].w);
                        }
                    }
                }
            }
        }
        // Smallest (distance, index) across the group.
#pragma unroll
        for (int o = ST_G / 2; o > 0; o >>= 1) {
            const int od = __shfl_xor(bestDist, o, ST_G), oi = __shfl_xor(bestIdx, o, ST_G);
            const float ou = __shfl_xor(bestU, o, ST_G);
            if (od < bestDist || (od == bestDist && oi < bestIdx)) {
                bestDist = od;
                bestIdx = oi;
                bestU = ou;
            }
        }
        go = bestDist < 75 && bestIdx != INT_MAX;
    }
    int sx0 = 0, sy0 = 0, sxR = 0;
    float scaleduR0 = 0.f;
    if (go) {
        const float uR0 = bestU;
        const float scaleFactor = A.inv_scale[levelL];
        const float scaleduL = roundf(uL * scaleFactor);
        const float scaledvL = roundf(vL * scaleFactor);
        scaleduR0 = roundf(uR0 * scaleFactor);
        const float iniu = scaleduR0 - 5 - 5;
        const float endu = scaleduR0 + 5 + 5 + 1;
        if (iniu < 0 || endu >= wR) go = false;
        sx0 = (int)scaleduL;
        sy0 = (int)scaledvL;
        sxR = (int)scaleduR0;
        // Keypoints of this extractor always leave room for the 11x11
        // patches; caller-supplied ones are checked instead of read past the
        // level (the reference would index outside the cv::Mat).
        if (sy0 - 5 < 0 || sy0 + 5 >= hL || sy0 + 5 >= hR || sx0 - 5 < 0 || sx0 + 5 >= wL) go = false;
    }
    if (go) {
        // Lane r < 11: patch row r, left bytes l0..l10 (x = sx0-5 ..) and
        // right bytes r0..r20 (x = sxR-10 ..); lanes 11..15 repeat row 10
        // and contribute nothing.
        const int r = sub < 11 ? sub : 10;
        const uint8_t* rl = pl + (unsigned)((sy0 - 5 + r) * pitchL);
        const uint8_t* rr = pr + (unsigned)((sy0 - 5 + r) * pitchR);
        const int xl0 = (sx0 - 5) & ~3, offL = sx0 - 5 - xl0;
        const int xr0 = (sxR - 10) & ~3, offR = sxR - 10 - xr0;
        unsigned dl[4], dr[6];
        if (xl0 + 15 < wL) {                     // the whole 16 bytes lie in the row
            const uint4 q = gload16(rl + xl0);
            dl[0] = q.x, dl[1] = q.y, dl[2] = q.z, dl[3] = q.w;
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++) dl[k] = patch_dword(rl, xl0 + 4 * k, wL);
        }
        if (xr0 + 23 < wR) {
            const uint4 q = gload16(rr + xr0);
            const uint2 q2 = gload8(rr + xr0 + 16);
            dr[0] = q.x, dr[1] = q.y, dr[2] = q.z, dr[3] = q.w, dr[4] = q2.x, dr[5] = q2.y;
        } else {
#pragma unroll
            for (int k = 0; k < 6; k++) dr[k] = patch_dword(rr, xr0 + 4 * k, wR);
        }
        unsigned la[3], ra[6];
#pragma unroll
        for (int k = 0; k < 3; k++) la[k] = __builtin_amdgcn_alignbyte(dl[k + 1], dl[k], (unsigned)offL);
#pragma unroll
        for (int k = 0; k < 5; k++) ra[k] = __builtin_amdgcn_alignbyte(dr[k + 1], dr[k], (unsigned)offR);
        ra[5] = dr[5] >> (8 * offR);
        // Centres from row 5: cL = l5, cR of shift s = r(s+5), s = 0..10.
        const int cL = __shfl((int)((la[1] >> 8) & 0xFFu), gbase + 5, 64);
        const unsigned c0 = (unsigned)__shfl((int)__builtin_amdgcn_alignbyte(ra[2], ra[1], 1u), gbase + 5, 64);
        const unsigned c1 = (unsigned)__shfl((int)__builtin_amdgcn_alignbyte(ra[3], ra[2], 1u), gbase + 5, 64);
        const unsigned c2 = (unsigned)__shfl((int)__builtin_amdgcn_alignbyte(ra[4], ra[3], 1u), gbase + 5, 64);
        // Left pairs (l2k, l2k+1), k < 5, and (l10, 0).
        unsigned lp[6];
#pragma unroll
        for (int k = 0; k < 5; k++) lp[k] = __builtin_amdgcn_perm(0u, la[k >> 1], (k & 1) ? 0x0C030C02u : 0x0C010C00u);
        lp[5] = (la[2] >> 16) & 0xFFu;
        // Right pairs (rj, rj+1) + 256 each, j < 20, and (rj, 0) + 256, j = 10..20.
        unsigned rp[20], rs[11];
#pragma unroll
        for (int j = 0; j < 20; j++) {
            const int q = j >> 2, p = j & 3;
            rp[j] = __builtin_amdgcn_perm(q + 1 < 6 ? ra[q + 1] : 0u, ra[q],
                                          0x0C000C00u | ((unsigned)(p + 1) << 16) | (unsigned)p) |
                    0x01000100u;
        }
#pragma unroll
        for (int j = 10; j <= 20; j++) rs[j - 10] = ((ra[j >> 2] >> (8 * (j & 3))) & 0xFFu) | 0x100u;
        unsigned part[11];
#pragma unroll
        for (int s = 0; s < 11; s++) {
            const unsigned cw = s < 4 ? c0 : (s < 8 ? c1 : c2);
            const unsigned e = ((cw >> (8 * (s & 3))) & 0xFFu) + 256u - (unsigned)cL;   // cR - cL + 256
            const unsigned e2 = e | (e << 16);
            unsigned acc = 0;
#pragma unroll
            for (int k = 0; k < 5; k++) acc = __builtin_amdgcn_sad_u16(lp[k] + e2, rp[s + 2 * k], acc);
            part[s] = __builtin_amdgcn_sad_u16(lp[5] + e, rs[s], acc);
        }
        unsigned tot[6];
#pragma unroll
        for (int m = 0; m < 6; m++) {
            const unsigned v = 2 * m + 1 < 11 ? (part[2 * m] | (part[2 * m + 1] << 16)) : part[2 * m];
            tot[m] = row16_sum(sub < 11 ? v : 0u);
        }
        int sad[11];
#pragma unroll
        for (int s = 0; s < 11; s++) sad[s] = (int)((tot[s >> 1] >> (16 * (s & 1))) & 0xFFFFu);
        // First minimum over inc = -5..5, then the parabola on its
        // neighbours, evaluated identically by every lane of the group.
        unsigned key = 0xFFFFFFFFu;
#pragma unroll
        for (int s = 0; s < 11; s++) key = min(key, ((unsigned)sad[s] << 4) | (unsigned)s);
        const int best = (int)(key >> 4), bs = (int)(key & 15u);
        const int bestinc = bs - 5;
        int d1 = 0, d3 = 0;
#pragma unroll
        for (int s = 0; s < 11; s++) {
            d1 = s == bs - 1 ? sad[s] : d1;
            d3 = s == bs + 1 ? sad[s] : d3;
        }
        if (bestinc != -5 && bestinc != 5) {
            const float dist1 = (float)d1;
            const float dist2 = (float)best;
            const float dist3 = (float)d3;
            const float deltaR = __fdiv_rn(dist1 - dist3, 2.0f * (dist1 + dist3 - 2.0f * dist2));
            if (!(deltaR < -1 || deltaR > 1)) {
                float bestuR = A.scale[levelL] * ((float)scaleduR0 + (float)bestinc + deltaR);
                float disparity = (uL - bestuR);
                if (disparity >= minD && disparity < maxD) {
                    if (disparity <= 0) {
                        disparity = 0.01f;
                        bestuR = (float)((double)uL - 0.01);
                    }
                    outD = __fdiv_rn(A.bf, disparity);
                    outU = bestuR;
                    outSad = best;
                }
            }
        }
    }
    if (sub == 0) {
        A.uRight[iL] = outU;
        A.depth[iL] = outD;
        A.match_sad[iL] = outSad;
    }
}

// Median cut (Frame.cc:1066-1081): matches whose SAD is not below
// 1.5 * 1.4 * median are dropped, the median being element M/2 of the M
// kept SADs in ascending order.  One workgroup per pair selects it with two
// 256-bin histograms (SADs are below 2^16), high byte then low byte, and
// clears the rejected keypoints.
#define MEDIAN_T 1024
#define MEDIAN_PER_T 4               // left keypoints per thread (<= 4096)

// Wavefront 0: the bin of s_h holding rank k (0-based) of the ascending
// order, and k's offset inside it; bin -1 when the histogram holds <= k.
__device__ __forceinline__ void median_pick(const int* s_h, int k, int* s_out)
{
    const int lane = threadIdx.x;
    int c[4], s = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        c[j] = s_h[4 * lane + j];
        s += c[j];
    }
    int inc = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(inc, o, 64);
        if (lane >= o) inc += v;
    }
    int ex = inc - s;
    if (lane == 63 && inc <= k) s_out[0] = -1;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (ex <= k && k < ex + c[j]) {
            s_out[0] = 4 * lane + j;
            s_out[1] = k - ex;
        }
        ex += c[j];
    }
}

__global__ __launch_bounds__(MEDIAN_T) void stereo_median_kernel(const StereoArgs* __restrict__ args)
{
    __shared__ int s_h[256];
    __shared__ int s_m;
    __shared__ int s_sel[2];
    const StereoArgs& A = args[blockIdx.x];
    const int t = threadIdx.x;
    const int n = min(min(*A.nl, A.cap_l), MEDIAN_T * MEDIAN_PER_T);
    if (t < 256) s_h[t] = 0;
    if (t == 0) s_m = 0;
    __syncthreads();
    int sad[MEDIAN_PER_T], m = 0;
#pragma unroll
    for (int k = 0; k < MEDIAN_PER_T; k++) {
        const int i = t + MEDIAN_T * k;
        sad[k] = i < n ? (int)gload4((const uint8_t*)(A.match_sad + i)) : -1;
        if (sad[k] >= 0) {
            atomicAdd(&s_h[sad[k] >> 8], 1);
            m++;
        }
    }
    if (m) atomicAdd(&s_m, m);
    __syncthreads();
    const int M = s_m;
    if (M == 0) return;                              // nothing to cut (uniform)
    if (t < 64) median_pick(s_h, M / 2, s_sel);
    __syncthreads();
    const int hb = s_sel[0], k2 = s_sel[1];
    __syncthreads();
    if (t < 256) s_h[t] = 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < MEDIAN_PER_T; k++)
        if (sad[k] >= 0 && (sad[k] >> 8) == hb) atomicAdd(&s_h[sad[k] & 255], 1);
    __syncthreads();
    if (t < 64) median_pick(s_h, k2, s_sel);
    __syncthreads();
    const float median = (float)((hb << 8) | s_sel[0]);
    const float kf = 1.5f * 1.4f;
    const float thDist = kf * median;
#pragma unroll
    for (int k = 0; k < MEDIAN_PER_T; k++) {
        const int i = t + MEDIAN_T * k;
        if (sad[k] >= 0 && !((float)sad[k] < thDist)) {
            gstore4((uint8_t*)(A.uRight + i), __float_as_uint(-1.0f));
            gstore4((uint8_t*)(A.depth + i), __float_as_uint(-1.0f));
        }
    }
}

// ============================================================ brute force
// Best/second-best Hamming match per query with the update rule of
// ORBmatcher::SearchForInitialization (ORBmatcher.cc:614-647): the best is
// the first minimum in index order, the second is the next-smallest distance
// in the multiset; accept iff best <= th_low and best < (float)second*ratio.
__global__ __launch_bounds__(256) void match_bf_kernel(const uint8_t* __restrict__ q, const int* __restrict__ nq_ptr,
                                                       const uint8_t* __restrict__ t, const int* __restrict__ nt_ptr,
                                                       int th_low, float ratio, int* __restrict__ idx,
                                                       int* __restrict__ dist, int cap_q)
{
    const int lane = threadIdx.x & 63;
    const int iq = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int nq = *nq_ptr, nt = *nt_ptr;
    if (iq >= nq || iq >= cap_q) return;
    const uint4 a0 = *(const uint4*)(q + (size_t)iq * 32);
    const uint4 a1 = *(const uint4*)(q + (size_t)iq * 32 + 16);
    int d0 = INT_MAX, i0 = INT_MAX, d1 = INT_MAX;
    for (int j = lane; j < nt; j += 64) {
        const int d = hamming32(a0, a1, t + (size_t)j * 32);
        if (d < d0) {
            d1 = d0;
            d0 = d;
            i0 = j;
        } else if (d < d1) {
            d1 = d;
        }
    }
    int bd = d0, bi = i0;
    for (int o = 32; o > 0; o >>= 1) {
        const int od = __shfl_xor(bd, o, 64), oi = __shfl_xor(bi, o, 64);
        if (od < bd || (od == bd && oi < bi)) {
            bd = od;
            bi = oi;
        }
    }
    int sec = (i0 == bi) ? d1 : d0;
    for (int o = 32; o > 0; o >>= 1) sec = min(sec, __shfl_xor(sec, o, 64));
    if (lane == 0) {
        const bool ok = bi != INT_MAX && bd <= th_low && (float)bd < (float)sec * ratio;
        idx[iq] = ok ? bi : -1;
        dist[iq] = bd;
    }
}

// Many (query set, train set) matches in one launch, one wavefront per query.
__device__ __forceinline__ int find_match(const MatchArgs* args, int n, int x)
{
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (args[mid].wave_base <= x) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

__global__ __launch_bounds__(256) void match_pairs_kernel(const MatchArgs* __restrict__ args, int npairs, int nwaves)
{
    const int lane = threadIdx.x & 63;
    const int wid = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (wid >= nwaves) return;
    const MatchArgs& A = args[find_match(args, npairs, wid)];
    const int iq = wid - A.wave_base;
    const int nq = *A.nq, nt = *A.nt;
    if (iq >= nq || iq >= A.cap_q) return;
    const uint4 a0 = *(const uint4*)(A.q + (size_t)iq * 32);
    const uint4 a1 = *(const uint4*)(A.q + (size_t)iq * 32 + 16);
    int d0 = INT_MAX, i0 = INT_MAX, d1 = INT_MAX;
    for (int j = lane; j < nt; j += 64) {
        const int d = hamming32(a0, a1, A.t + (size_t)j * 32);
        if (d < d0) {
            d1 = d0;
            d0 = d;
            i0 = j;
        } else if (d < d1) {
            d1 = d;
        }
    }
    int bd = d0, bi = i0;
    for (int o = 32; o > 0; o >>= 1) {
        const int od = __shfl_xor(bd, o, 64), oi = __shfl_xor(bi, o, 64);
        if (od < bd || (od == bd && oi < bi)) {
            bd = od;
            bi = oi;
        }
    }
    int sec = (i0 == bi) ? d1 : d0;
    for (int o = 32; o > 0; o >>= 1) sec = min(sec, __shfl_xor(sec, o, 64));
    if (lane == 0) {
        const bool ok = bi != INT_MAX && bd <= A.th_low && (float)bd < (float)sec * A.ratio;
        A.idx[iq] = ok ? bi : -1;
        A.dist[iq] = bd;
    }
}

// After the matches of a launch: each pair's query rows become the resident
// "previous" set of its stream (one workgroup per pair).
__global__ __launch_bounds__(256) void save_prev_kernel(const MatchArgs* __restrict__ args, int npairs)
{
    const MatchArgs& A = args[blockIdx.x];
    if (!A.save_desc) return;
    const int n = min(*A.nq, A.save_cap);
    const uint4* src = (const uint4*)A.q;
    uint4* dst = (uint4*)A.save_desc;
    for (int i = threadIdx.x; i < 2 * n; i += 256) dst[i] = src[i];
    if (threadIdx.x == 0) *A.save_n = n;
}

// ============================================================= launchers
// ev (optional): events recorded after each stage -- [0] start, then one per
// pyramid level (max_levels; level 1 with the resize of all levels), octree,
// describe.  Without events the levels' tiles are one launch.
extern "C" hipError_t orb_launch_extract(const ImageJob* d_jobs, const RunTable* d_rt, const RunTable* h_rt,
                                         hipStream_t st, hipEvent_t* ev)
{
    int e = 0;
    if (ev) (void)hipEventRecord(ev[e++], st);
    auto pyramid = [&](int zero) {
        for (int c = 0; c < h_rt->nchains; c++) {
            const int nb = h_rt->chain_start[c][h_rt->njobs];
            if (nb <= 0) continue;
            if (h_rt->chain_variant == 0)
                pyramid_kernel<0><<<nb, ORB_CH_T, 0, st>>>(d_jobs, d_rt, c, c == 0 ? zero : 0);
            else
                pyramid_kernel<1><<<nb, ORB_CH_T, 0, st>>>(d_jobs, d_rt, c, c == 0 ? zero : 0);
        }
    };
    auto tiles = [&](int th, int level) {
        const int nb = level < 0 ? h_rt->all_start[th == 16 ? 1 : 0][h_rt->max_levels]
                                 : h_rt->tile_start[level][h_rt->njobs];
        if (nb <= 0) return;
        if (th == 16) level_kernel<16><<<nb, 256, 0, st>>>(d_jobs, d_rt, level);
        else level_kernel<32><<<nb, 256, 0, st>>>(d_jobs, d_rt, level);
    };
    if (ev || !h_rt->chain_zeroes) zero_counters_kernel<<<h_rt->njobs, 256, 0, st>>>(d_jobs, h_rt->njobs);
    if (!ev) {
        pyramid(h_rt->chain_zeroes);
        tiles(32, -1);
        tiles(16, -1);
    } else {
        // stage by stage: level 0, then the pyramid with level 1, then the others
        for (int l = 0; l < h_rt->max_levels; l++) {
            if (l == 1) pyramid(0);
            tiles(h_rt->tile_h[l], l);
            (void)hipEventRecord(ev[e++], st);
        }
    }
    octree_kernel<<<h_rt->njobs * h_rt->max_levels, OCT_T, 0, st>>>(d_jobs, h_rt->max_levels);
    if (ev) (void)hipEventRecord(ev[e++], st);
    const int nblocks = h_rt->desc_start[h_rt->njobs * h_rt->max_levels];
    if (nblocks > 0) describe_kernel<<<nblocks, 256, 0, st>>>(d_jobs, d_rt);
    if (ev) (void)hipEventRecord(ev[e++], st);
    return hipGetLastError();
}

// d_args: npairs StereoArgs in device memory; max_left: the largest cap_l.
// ev (optional): events after the match kernel and after the median cut.
extern "C" hipError_t orb_launch_stereo(const StereoArgs* d_args, int npairs, int max_left, hipStream_t st,
                                        hipEvent_t* ev)
{
    if (npairs <= 0) return hipSuccess;
    stereo_prep_kernel<<<npairs, 1024, 0, st>>>(d_args);
    if (max_left > 0) stereo_kernel<<<dim3((max_left + 256 / ST_G - 1) / (256 / ST_G), npairs), 256, 0, st>>>(d_args);
    if (ev) (void)hipEventRecord(ev[0], st);
    stereo_median_kernel<<<npairs, 1024, 0, st>>>(d_args);
    if (ev) (void)hipEventRecord(ev[1], st);
    return hipGetLastError();
}

extern "C" hipError_t orb_launch_match_bf(const uint8_t* q, const int* nq, const uint8_t* t, const int* nt,
                                          int th_low, float ratio, int* idx, int* dist, int cap_q,
                                          hipStream_t st)
{
    if (cap_q > 0) match_bf_kernel<<<(cap_q + 3) / 4, 256, 0, st>>>(q, nq, t, nt, th_low, ratio, idx, dist, cap_q);
    return hipGetLastError();
}

// ============================================================ dense k=2
// All-pairs Hamming search of nq queries against nm map rows, k = 2 nearest
// by (distance, index), the order of ORBmatcher's best/second-best update
// (ORBmatcher.cc:614-647).  The map is split into chunks of at most KNN_CHUNK
// rows; each (chunk, query block) workgroup keeps two keys per query
//   key = distance << 20 | row-in-chunk
// (lexicographic (distance, index) is numeric key order), and a merge kernel
// reduces the chunks:
//   knn_popc_kernel  XOR + v_bcnt popcount, one query per lane, map rows
//                    broadcast from LDS; the keys are the chunk's two
//                    smallest
//   knn_mfma_kernel  bits expanded to FP4, the distance a sum of exact
//                    products on the matrix cores; the keys are the two
//                    smallest of the minima of groups of 16 rows, and the
//                    merge looks at the best row's group
#define KNN_CHUNK 8192
#define KNN_NONE 0xFFFFFFFFu
#ifndef KNN_NG
#define KNN_NG 2                     // 32-query groups per wavefront (4: 1 % faster at 2000 x 1M, slower below)
#endif

// Median of three (the compiler emits v_med3_u32 / v_med3_i32).
__device__ __forceinline__ unsigned med3u(unsigned a, unsigned b, unsigned c)
{
    return max(min(a, b), min(max(a, b), c));
}

__device__ __forceinline__ int med3i(int a, int b, int c)
{
    return max(min(a, b), min(max(a, b), c));
}

__global__ __launch_bounds__(256) void knn_popc_kernel(const uint8_t* __restrict__ q, int nq,
                                                       const uint8_t* __restrict__ m, long long nm,
                                                       uint2* __restrict__ part, int nchunks, int chunk_rows)
{
    __shared__ uint4 rows[256][2];
    const int tid = threadIdx.x;
    const int chunk = blockIdx.x;
    const int qi = blockIdx.y * 256 + tid;
    uint4 a0 = make_uint4(0, 0, 0, 0), a1 = a0;
    if (qi < nq) {
        a0 = *(const uint4*)(q + (size_t)qi * 32);
        a1 = *(const uint4*)(q + (size_t)qi * 32 + 16);
    }
    const long long c0 = (long long)chunk * chunk_rows;
    const int len = (int)min((long long)chunk_rows, nm - c0);
    unsigned k0 = KNN_NONE, k1 = KNN_NONE;
    for (int t0 = 0; t0 < len; t0 += 256) {
        const int n = min(256, len - t0);
        __syncthreads();
        if (tid < n) {
            const uint8_t* r = m + (size_t)(c0 + t0 + tid) * 32;
            rows[tid][0] = *(const uint4*)r;
            rows[tid][1] = *(const uint4*)(r + 16);
        }
        __syncthreads();
        for (int r = 0; r < n; r++) {
            const uint4 b0 = rows[r][0], b1 = rows[r][1];
            unsigned d = __popc(a0.x ^ b0.x);
            d += __popc(a0.y ^ b0.y);
            d += __popc(a0.z ^ b0.z);
            d += __popc(a0.w ^ b0.w);
            d += __popc(a1.x ^ b1.x);
            d += __popc(a1.y ^ b1.y);
            d += __popc(a1.z ^ b1.z);
            d += __popc(a1.w ^ b1.w);
            const unsigned key = (d << 20) | (unsigned)(t0 + r);
            k1 = med3u(k0, k1, key);
            k0 = min(k0, key);
        }
    }
    if (qi < nq) part[(size_t)qi * nchunks + chunk] = make_uint2(k0, k1);
}

typedef int knn_v8i __attribute__((ext_vector_type(8)));
typedef float knn_v16f __attribute__((ext_vector_type(16)));

// Bit -> FP4 (E2M1) expansion of a descriptor word into the 32 nibbles of
// one MFMA operand lane: nibble k of dword i holds bit 4k + i.  Map side: a
// clear bit is 0 and a set bit 0.5, 1, 2 and 2 in dwords 0 .. 3 (the code's
// bits 0, 1, 2 and 2, so that three of the four dwords are one mask each).
// Query side: +-2, 1, 0.5 and 0.5, minus for a set bit, so every product is
// 0 or +-1.  Both sides use the same order, so the hardware's own k order
// cancels.
__device__ __forceinline__ knn_v8i expand_map(unsigned w)
{
    return (knn_v8i){(int)(w & 0x11111111u), (int)(w & 0x22222222u), (int)(w & 0x44444444u),
                     (int)((w >> 1) & 0x44444444u), 0, 0, 0, 0};
}

__device__ __forceinline__ knn_v8i expand_query(unsigned w)
{
    return (knn_v8i){(int)(((w << 3) & 0x88888888u) | 0x44444444u), (int)(((w << 2) & 0x88888888u) | 0x22222222u),
                     (int)(((w << 1) & 0x88888888u) | 0x11111111u), (int)((w & 0x88888888u) | 0x11111111u), 0, 0, 0, 0};
}

// Workgroup: 4 wavefronts, the same 32 * NG queries, one map chunk; wavefront
// w takes the 32-row tiles w, w + 4, ...  Bound: the MFMA pipe (a kernel of
// the same instructions on registers alone reaches 7.5 of the 10 POP/s).
// 2000 queries x 1M rows: search 184 us (5.6 POP/s), a call among others 178
// where int8 MFMAs with every key kept took 402; 64 x 1M 14 us (171).
//
// v_mfma_scale_f32_32x32x64_f8f6f4 on FP4 operands does 65536 multiply-adds
// in 32 cycles, twice the int8 rate, and a descriptor word expands into one
// operand lane with 5 VALU ops.  sum m (1 - 2q) = Hamming - |q|; the C input
// adds 256 and the row / 8192, so every accumulator is a non-negative
// multiple of 2^-13 below 513, of at most 23 bits (an empty query against a
// full row), exact in float, and its bits order as an integer:
//   key = Hamming - |q| + 256 + row / 8192.
// |q| is constant per query, so keys order (distance, row).
//
// The 16 accumulators of a lane are 16 rows of one tile for one query.  Only
// the smallest is kept (8 v_min3 for 16 keys) and enters the lane's two
// smallest: of all such groups of 16 rows, the best row is the minimum of
// the group with the smallest minimum, and the second best is either the
// next group's minimum or in the best row's own group, whose other 15 rows
// the merge kernel looks at.  That is 11 VALU ops for 16 keys where keeping
// the two smallest of all keys takes 32.
template <int NG>
__global__ __launch_bounds__(256) void knn_mfma_kernel(const uint8_t* __restrict__ q, int nq,
                                                       const uint8_t* __restrict__ m, long long nm,
                                                       uint2* __restrict__ part, int nchunks, int chunk_rows)
{
    __shared__ int2 s_key[3][NG][64];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int hb = lane >> 5, i32 = lane & 31;
    // XCD x (workgroups b with b % 8 == x; a row of the grid is a multiple of
    // 8 of them) takes chunks x, x + 8, ..., a grid row's chunks' query blocks
    // one after another, so a chunk's rows come from memory once and from that
    // XCD's L2 after that (2000 x 1M search 220 -> 197 us against chunks spread
    // over the XCDs).
    const int chunk = (int)(blockIdx.y * ORB_NUM_XCD + blockIdx.x % ORB_NUM_XCD);
    const int qbase = (int)(blockIdx.x / ORB_NUM_XCD) * 32 * NG;
    if (chunk >= nchunks) return;

    // Query operands: lane (query i32, half hb) holds words 4 hb + c.
    knn_v8i B[NG][4];
    int pop[NG];
#pragma unroll
    for (int n = 0; n < NG; n++) {
        const int qi = min(qbase + 32 * n + i32, nq - 1);
        const uint4 w = gload16(q + (size_t)qi * 32 + 16 * hb);
        B[n][0] = expand_query(w.x);
        B[n][1] = expand_query(w.y);
        B[n][2] = expand_query(w.z);
        B[n][3] = expand_query(w.w);
        pop[n] = __popc(w.x) + __popc(w.y) + __popc(w.z) + __popc(w.w);
        pop[n] += __shfl_xor(pop[n], 32, 64);
    }
    const long long c0 = (long long)chunk * chunk_rows;
    const int len = (int)min((long long)chunk_rows, nm - c0);
    int k0[NG], k1[NG];
#pragma unroll
    for (int n = 0; n < NG; n++) k0[n] = k1[n] = INT_MAX;
    // Accumulator r of a lane is row 8 (r >> 2) + 4 hb + (r & 3) of the tile.
    knn_v16f rows;
#pragma unroll
    for (int r = 0; r < 16; r++) rows[r] = 256.f + (float)(8 * (r >> 2) + 4 * hb + (r & 3)) * (1.f / KNN_CHUNK);

    const uint8_t* mchunk = m + (size_t)c0 * 32;
    // Rows past the chunk's end read its last row; their keys are discarded.
    auto load = [&](int t0) {
        return gload16(mchunk + ((unsigned)min(t0 + i32, len - 1) * 32u + 16u * (unsigned)hb));
    };
    uint4 wn = load(min(32 * wv, len - 1));
    for (int t0 = 32 * wv; t0 < len; t0 += 128) {
        const knn_v8i A[4] = {expand_map(wn.x), expand_map(wn.y), expand_map(wn.z), expand_map(wn.w)};
        if (t0 + 128 < len) wn = load(t0 + 128);
        knn_v16f acc[NG];
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int n = 0; n < NG; n++)
                acc[n] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(A[c], B[n][c], c == 0 ? rows : acc[n], 4, 4, 0, 0,
                                                                        0, 0);
        if (t0 + 32 > len) {                       // the chunk's last, partial tile
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const bool ok = t0 + 8 * (r >> 2) + 4 * hb + (r & 3) < len;
#pragma unroll
                for (int n = 0; n < NG; n++) acc[n][r] = ok ? acc[n][r] : __int_as_float(0x7F000000);
            }
        }
        const float tile = (float)t0 * (1.f / KNN_CHUNK);
#pragma unroll
        for (int n = 0; n < NG; n++) {
            int g = __float_as_int(acc[n][0]);
#pragma unroll
            for (int r = 1; r < 16; r++) g = min(g, __float_as_int(acc[n][r]));
            const int key = __float_as_int(__int_as_float(g) + tile);
            k1[n] = med3i(k0[n], k1[n], key);
            k0[n] = min(k0[n], key);
        }
    }
    // Merge the two lanes that hold a query, then the four wavefronts.
#pragma unroll
    for (int n = 0; n < NG; n++) {
        const int b0 = __shfl_xor(k0[n], 32, 64), b1 = __shfl_xor(k1[n], 32, 64);
        const int n0 = min(k0[n], b0);
        k1[n] = min(max(k0[n], b0), min(k1[n], b1));
        k0[n] = n0;
        if (wv > 0) s_key[wv - 1][n][lane] = make_int2(k0[n], k1[n]);
    }
    __syncthreads();
    if (wv == 0 && hb == 0) {
#pragma unroll
        for (int n = 0; n < NG; n++) {
#pragma unroll
            for (int w = 0; w < 3; w++) {
                const int2 o = s_key[w][n][lane];
                const int n0 = min(k0[n], o.x);
                k1[n] = min(max(k0[n], o.x), min(k1[n], o.y));
                k0[n] = n0;
            }
            const int qi = qbase + 32 * n + i32;
            if (qi < nq) {
                const int ks[2] = {k0[n], k1[n]};
                unsigned out[2];
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    // keys of rows past the end are at least 2^127
                    const int v = ks[t] < 0x7F000000 ? (int)(__int_as_float(ks[t]) * KNN_CHUNK) : 0;
                    out[t] = ks[t] >= 0x7F000000
                                 ? KNN_NONE
                                 : ((unsigned)((v >> 13) - 256 + pop[n]) << 20) | (unsigned)(v & (KNN_CHUNK - 1));
                }
                part[(size_t)qi * nchunks + chunk] = make_uint2(out[0], out[1]);
            }
        }
    }
}

// Reduce the per-chunk keys of each query to the global two nearest and apply
// the ratio test (best < ratio * second, in float).  A wavefront per query:
// its lanes stride over the chunks, then 16 of them take a row each of the
// best row's group (knn_mfma_kernel keeps one key per group of 16).  knn_popc_kernel's keys are
// the two smallest already, and then the group holds none nearer.  Bound:
// latency; 4 us for 2000 queries x 123 chunks, where one thread per query
// took 47 us, a chain of scattered reads.
__global__ __launch_bounds__(256) void knn_merge_kernel(const uint2* __restrict__ part, int nq, int nchunks,
                                                        int chunk_rows, const uint8_t* __restrict__ q,
                                                        const uint8_t* __restrict__ m, long long nm, float ratio,
                                                        int* __restrict__ idx2, int* __restrict__ dist2,
                                                        uint8_t* __restrict__ accept)
{
    const int lane = threadIdx.x & 63, sub = lane & 15;
    const int qi = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (qi >= nq) return;                          // the whole wavefront leaves
    unsigned long long b0 = ~0ull, b1 = ~0ull;     // distance << 40 | row
    auto take = [&](unsigned long long k) {
        b1 = k < b0 ? b0 : (k < b1 ? k : b1);
        b0 = k < b0 ? k : b0;
    };
    for (int c = lane; c < nchunks; c += 64) {
        const uint2 p = part[(size_t)qi * nchunks + c];
        const unsigned ks[2] = {p.x, p.y};
#pragma unroll
        for (int t = 0; t < 2; t++)
            if (ks[t] != KNN_NONE)
                take(((unsigned long long)(ks[t] >> 20) << 40) |
                     (unsigned long long)((long long)c * chunk_rows + (ks[t] & 0xFFFFF)));
    }
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long c0 = __shfl_xor(b0, o, 64), c1 = __shfl_xor(b1, o, 64);
        const unsigned long long n0 = min(b0, c0);
        b1 = min(max(b0, c0), min(b1, c1));
        b0 = n0;
    }
    if (b0 != ~0ull) {
        const long long best = (long long)(b0 & 0xFFFFFFFFFFull);
        const long long row = (best & ~31ll) + 8 * (sub >> 2) + (best & 4) + (sub & 3);
        unsigned long long k = ~0ull;
        if (row < nm && row != best) {
            const uint4 a0 = *(const uint4*)(q + (size_t)qi * 32), a1 = *(const uint4*)(q + (size_t)qi * 32 + 16);
            k = ((unsigned long long)hamming32(a0, a1, m + (size_t)row * 32) << 40) | (unsigned long long)row;
        }
        for (int o = 1; o < 16; o <<= 1) k = min(k, __shfl_xor(k, o, 16));
        b1 = min(b1, k);
    }
    if (lane != 0) return;
    const int d0 = b0 == ~0ull ? INT_MAX : (int)(b0 >> 40), d1 = b1 == ~0ull ? INT_MAX : (int)(b1 >> 40);
    idx2[2 * qi] = b0 == ~0ull ? -1 : (int)(b0 & 0xFFFFFFFFFFull);
    idx2[2 * qi + 1] = b1 == ~0ull ? -1 : (int)(b1 & 0xFFFFFFFFFFull);
    dist2[2 * qi] = d0;
    dist2[2 * qi + 1] = d1;
    if (accept) accept[qi] = (uint8_t)(b0 != ~0ull && b1 != ~0ull && (float)d0 < (float)d1 * ratio);
}

// Rows per map chunk: KNN_CHUNK, halved while the grid has fewer than 1024
// workgroups (the GPU holds that many), down to 512 rows, as long as the
// partial keys (one entry per query and chunk) stay within max_entries.
// Search + merge in us at 8192, 4096, 2048 and 512 rows: 500 x 100k 23 + 6, 15
// + 6, 12 + 6, 13 + 7; 2000 x 1M 186 + 7, 187 + 8, 197 + 10, 258 + 21; 64 x 1M
// 24 + 6, 15 + 7, 13 + 9, 14 + 18 (the merge grows with the chunks).
extern "C" int orb_knn_chunk_rows(int nq, long long nm, int method, size_t max_entries)
{
    const long long tiles = method == 1 ? (nq + 32 * KNN_NG - 1) / (32 * KNN_NG) : (nq + 255) / 256;
    int rows = KNN_CHUNK;
    while (rows > 512 && tiles * ((nm + rows - 1) / rows) < 1024 &&
           (unsigned long long)nq * (unsigned long long)((nm + rows / 2 - 1) / (rows / 2)) <= max_entries)
        rows /= 2;
    return rows;
}

// The MFMA search's grid: query blocks (8 workgroups each, a chunk apiece) by
// groups of 8 chunks.  HIP wants fewer than 2^32 threads along x and 65536
// workgroups along y: at most 2^27 queries, and 2^31 rows are 2^15 groups of
// KNN_CHUNK rows (smaller chunks are for grids below 1024 workgroups).
// Returns 0, or -1 where the grid does not fit.
extern "C" int orb_knn_grid(int nq, long long nm, int chunk_rows, unsigned* x, unsigned* y)
{
    const long long chunks = (nm + chunk_rows - 1) / chunk_rows;
    const long long gx = ORB_NUM_XCD * (((long long)nq + 32 * KNN_NG - 1) / (32 * KNN_NG));
    const long long gy = (chunks + ORB_NUM_XCD - 1) / ORB_NUM_XCD;
    if (gx * 256 >= (1ll << 32) || gy > 65535) return -1;
    *x = (unsigned)gx;
    *y = (unsigned)gy;
    return 0;
}

extern "C" hipError_t orb_launch_knn2(const uint8_t* q, int nq, const uint8_t* m, long long nm, int method,
                                      float ratio, uint2* part, int chunk_rows, int* idx2, int* dist2,
                                      uint8_t* accept, hipStream_t st, hipEvent_t* ev)
{
    const int nchunks = (int)((nm + chunk_rows - 1) / chunk_rows);
    if (nq <= 0) return hipSuccess;
    if (ev) (void)hipEventRecord(ev[0], st);
    if (nchunks > 0) {
        unsigned gx = 0, gy = 0;
        if (method == 1 && orb_knn_grid(nq, nm, chunk_rows, &gx, &gy)) return hipErrorInvalidValue;
        if (method == 1)
            knn_mfma_kernel<KNN_NG><<<dim3(gx, gy), 256, 0, st>>>(q, nq, m, nm, part, nchunks, chunk_rows);
        else
            knn_popc_kernel<<<dim3(nchunks, (nq + 255) / 256), 256, 0, st>>>(q, nq, m, nm, part, nchunks, chunk_rows);
    }
    if (ev) (void)hipEventRecord(ev[1], st);
    knn_merge_kernel<<<(nq + 3) / 4, 256, 0, st>>>(part, nq, nchunks, chunk_rows, q, m, nm, ratio, idx2, dist2, accept);
    if (ev) (void)hipEventRecord(ev[2], st);
    return hipGetLastError();
}

// ================================================= allocation-free dense k=2
// orb_knn2_device_noalloc keeps the per-chunk partial keys in this fixed
// array instead of a context buffer, so that it makes no allocation.  Each
// GPU holds its own copy until the process ends; host code uses the address
// orb_knn_scratch_setup looked up for the device, never the symbol itself.
#define ORB_KNN_SCRATCH_ENTRIES (1 << 19)   // uint2 keys: 4 MiB per GPU
#define ORB_KNN_SCRATCH_DEVICES 64
static __device__ __align__(256) uint2 scratch[ORB_KNN_SCRATCH_ENTRIES];
static uint2* g_scratch_ptr[ORB_KNN_SCRATCH_DEVICES];

// With `device` current: look up this GPU's copy of the array (once).
// Returns 0, or a HIP error code.
extern "C" int orb_knn_scratch_setup(int device)
{
    if (device < 0 || device >= ORB_KNN_SCRATCH_DEVICES) return (int)hipErrorInvalidDevice;
    if (__atomic_load_n(&g_scratch_ptr[device], __ATOMIC_ACQUIRE)) return 0;
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (!ptr) return (int)hipErrorInvalidSymbol;
    __atomic_store_n(&g_scratch_ptr[device], (uint2*)ptr, __ATOMIC_RELEASE);
    return 0;
}

// The device address of `device`'s array (null before its setup) and the
// number of uint2 keys it holds.
extern "C" uint2* orb_knn_scratch(int device, size_t* entries)
{
    if (entries) *entries = ORB_KNN_SCRATCH_ENTRIES;
    if (device < 0 || device >= ORB_KNN_SCRATCH_DEVICES) return nullptr;
    return __atomic_load_n(&g_scratch_ptr[device], __ATOMIC_ACQUIRE);
}

extern "C" hipError_t orb_launch_match_pairs(const MatchArgs* d_args, int npairs, int nwaves, hipStream_t st)
{
    if (npairs <= 0) return hipSuccess;
    if (nwaves > 0) match_pairs_kernel<<<(nwaves + 3) / 4, 256, 0, st>>>(d_args, npairs, nwaves);
    save_prev_kernel<<<npairs, 256, 0, st>>>(d_args, npairs);
    return hipGetLastError();
}

// ================================================== batch staged transfers
// One launch for a list of regions (blockIdx.y = region): a batch's pinned
// input images, landed in one device staging buffer by one host-to-device
// copy, go to their slots' images; the slots' outputs go into one buffer
// for one device-to-host copy.  A region whose length is a count read on the
// device copies only the valid entries.
// copy_list_kernel takes the list as an argument: a single call's counters,
// keypoints, descriptors and depths go straight into pinned host memory in one
// launch after the pipeline, so the call waits once and copies from there (it
// waited for the counts, then for a pageable copy per array).  Bound: latency.
// A call on 640 x 480 226 us before, 178 after; a stereo frame of 1241 x 376 428
// and 312, an RGB-D frame of 640 x 480 360 and 267; a batch of 64 pairs, its run
// and the read of all results, 4.71 ms (a copy per array) and 1.62.
__device__ __forceinline__ void copy_op(const CopyOp& o)
{
    int n = o.words;
    if (o.count) n = min(n, max(0, *o.count) * o.unit_words);
    const int stride = gridDim.x * 256;
    int i = blockIdx.x * 256 + threadIdx.x;
    if ((((uintptr_t)o.src | (uintptr_t)o.dst) & 15) == 0) {
        const int n4 = n >> 2;
        if (i < (n & 3)) o.dst[4 * n4 + i] = o.src[4 * n4 + i];
        for (; i < n4; i += stride) ((uint4*)o.dst)[i] = ((const uint4*)o.src)[i];
    } else {
        for (; i < n; i += stride) o.dst[i] = o.src[i];
    }
}

__global__ __launch_bounds__(256) void copy_ops_kernel(const CopyOp* __restrict__ ops) { copy_op(ops[blockIdx.y]); }

__global__ __launch_bounds__(256) void copy_list_kernel(const CopyList list) { copy_op(list.op[blockIdx.y]); }

extern "C" hipError_t orb_launch_copy_ops(const CopyOp* d_ops, int nops, int blocks_per_op, hipStream_t st)
{
    if (nops <= 0) return hipSuccess;
    copy_ops_kernel<<<dim3(blocks_per_op, nops), 256, 0, st>>>(d_ops);
    return hipGetLastError();
}

extern "C" hipError_t orb_launch_copy_list(const CopyList* list, int blocks_per_op, hipStream_t st)
{
    if (list->n <= 0) return hipSuccess;
    copy_list_kernel<<<dim3(blocks_per_op, list->n), 256, 0, st>>>(*list);
    return hipGetLastError();
}

// ======================================================= HBM copy microbench
// Plain streaming copy (16-byte loads and stores, grid-stride): the measured
// HBM rate of this kernel re-confirms the bandwidth peak, and its counter
// readings calibrate FETCH_SIZE / WRITE_SIZE for a known byte count.
__global__ __launch_bounds__(256) void hbm_copy_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                       size_t n16)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += stride) dst[i] = src[i];
}

extern "C" hipError_t orb_launch_hbm_copy(const void* src, void* dst, size_t bytes, hipStream_t st)
{
    const size_t n16 = bytes / 16;
    hbm_copy_kernel<<<8192, 256, 0, st>>>((const uint4*)src, (uint4*)dst, n16);
    return hipGetLastError();
}
