// orb_mappoint.hip -- MapPoint::ComputeDistinctiveDescriptors
// (src/MapPoint.cc:365-450) for many map points in one launch.
//
// The reference fills the N x N distance matrix,
// sorts every row (the zero self-distance included) and takes element
// (size_t)(0.5*(N-1)); the first row with the smallest such median wins.
// The median is the smallest v with #{j : d(i, j) <= v} >= (N-1)/2 + 1, found
// by binary search over v in [0, 256] -- the same order statistic without a
// sort.
//   N <= 128: lane i holds row i of the matrix, two 16-bit distances a
//   register, and searches its own row's median: 16 + 1 ops per column and
//   9 x 1.5 per distance serve 64 rows at once; one wavefront per point up to
//   N = 64, two beyond.  Bound: VALU and the scalar loads of the columns.
//   4000 points of 2..40 observations 18 us (106 row by row), 20000 66 (310).
//   N > 128: row by row, lane j holding d(i, j) for j = lane + 64c (c < 16, so
//   up to 1024 observations), with ballot counts, as a lane's row no longer
//   fits its registers; a workgroup per point.  300 points of
//   129..200 observations 102 us (485 with one wavefront each), of 65..128
//   26 us (258).
#include <hip/hip_runtime.h>
#include <stdint.h>

#define MP_MAX_CHUNKS 16             // 16 x 64 = 1024 observations per point

typedef unsigned short mp_us2 __attribute__((ext_vector_type(2)));

// Median of row `row` (each lane its own) for N <= 8 * NC observations, as a
// key median << 10 | row; rows past N give the largest key.  NC column blocks
// of 8; those past N are skipped.
template <int NC>
__device__ __forceinline__ int row_medians(const uint4* __restrict__ rows, int N, int need, int row)
{
    const int i = min(row, N - 1);
    const uint4 r0 = rows[2 * i], r1 = rows[2 * i + 1];
    unsigned d[4 * NC];                        // two distances each; 0xFFFF past N: never counted
#pragma unroll
    for (int c = 0; c < NC; c++) {
        if (8 * c < N) {
#pragma unroll
            for (int k = 0; k < 8; k++) {
                const int j = 8 * c + k, jr = min(j, N - 1);
                const uint4 q0 = rows[2 * jr], q1 = rows[2 * jr + 1];     // the same row for every lane
                unsigned x = __popc(r0.x ^ q0.x) + __popc(r0.y ^ q0.y) + __popc(r0.z ^ q0.z) + __popc(r0.w ^ q0.w) +
                             __popc(r1.x ^ q1.x) + __popc(r1.y ^ q1.y) + __popc(r1.z ^ q1.z) + __popc(r1.w ^ q1.w);
                x = j < N ? x : 0xFFFFu;
                if (k & 1) d[4 * c + (k >> 1)] |= x << 16;
                else d[4 * c + (k >> 1)] = x;
            }
        } else {
#pragma unroll
            for (int k = 0; k < 4; k++) d[4 * c + k] = 0xFFFFFFFFu;
        }
    }
    // (1 | 1 << 16 hidden from the optimiser, which otherwise turns the clamp
    // below into compares and selects of each half)
    unsigned one2 = 0x00010001u;
    asm volatile("" : "+s"(one2));
    int lo = 0, hi = 256;
#pragma unroll 1
    for (int step = 0; step < 9; step++) {
        const int mid = (lo + hi) >> 1;
        const unsigned t2 = (unsigned)(mid + 1) * 0x10001u;
        const mp_us2 t = __builtin_bit_cast(mp_us2, t2), one = __builtin_bit_cast(mp_us2, one2);
        mp_us2 cnt = {0, 0};
#pragma unroll
        for (int c = 0; c < NC; c++) {
            if (8 * c < N) {
#pragma unroll
                for (int k = 0; k < 4; k++)    // 1 where d < mid + 1
                    cnt += __builtin_elementwise_min(
                        __builtin_elementwise_sub_sat(t, __builtin_bit_cast(mp_us2, d[4 * c + k])), one);
            }
        }
        if (lo < hi) {
            if ((int)cnt.x + (int)cnt.y >= need) hi = mid;
            else lo = mid + 1;
        }
    }
    return row < N ? (lo << 10) | row : 0x7FFFFFFF;
}

__global__ __launch_bounds__(256) void distinctive_kernel(const uint8_t* __restrict__ desc,
                                                          const int* __restrict__ offsets, int n_points,
                                                          int* __restrict__ best, uint8_t* __restrict__ out_desc)
{
    const int lane = threadIdx.x & 63;
    const int p = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (p >= n_points) return;
    const int a = offsets[p], N = offsets[p + 1] - a;
    if (N > 64) return;                        // distinctive_large_kernel's
    if (N <= 0) {                              // no observation: -1 and a zero row
        if (lane == 0) best[p] = -1;
        if (out_desc && lane < 2) ((uint4*)(out_desc + (size_t)p * 32))[lane] = make_uint4(0, 0, 0, 0);
        return;
    }
    const int need = (N - 1) / 2 + 1;          // rank of the median, 1-based
    const uint4* rows = (const uint4*)(desc + (size_t)a * 32);
    int key = N <= 16 ? row_medians<2>(rows, N, need, lane)
                      : (N <= 32 ? row_medians<4>(rows, N, need, lane) : row_medians<8>(rows, N, need, lane));
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) key = min(key, __shfl_xor(key, o, 64));
    const int idx = key & 1023;
    if (lane == 0) best[p] = idx;
    if (out_desc && lane < 2) ((uint4*)(out_desc + (size_t)p * 32))[lane] = rows[2 * idx + lane];
}

// Points of more than 64 observations, one workgroup each (the others are
// passed over).  A kernel of its own: its registers (16 column blocks a row)
// would halve the wavefronts of the kernel above.
__global__ __launch_bounds__(256) void distinctive_large_kernel(const uint8_t* __restrict__ desc,
                                                                const int* __restrict__ offsets, int n_points,
                                                                int* __restrict__ best,
                                                                uint8_t* __restrict__ out_desc)
{
    __shared__ int s_key[4];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int p = blockIdx.x; p < n_points; p += gridDim.x) {
        const int a = offsets[p], N = offsets[p + 1] - a;
        if (N <= 64) continue;
        const int need = (N - 1) / 2 + 1;
        const uint4* rows = (const uint4*)(desc + (size_t)a * 32);
        int key = 0x7FFFFFFF;
        if (N <= 128) {                        // wavefronts 0 and 1: a row per lane
            if (wv < 2) key = row_medians<16>(rows, N, need, lane + 64 * wv);
        } else {                               // a wavefront per row, rows wv, wv + 4, ...
            const int nc = (N + 63) >> 6;
            for (int i = wv; i < N; i += 4) {
                const uint4 r0 = rows[2 * i], r1 = rows[2 * i + 1];
                int d[MP_MAX_CHUNKS];
#pragma unroll
                for (int c = 0; c < MP_MAX_CHUNKS; c++) {
                    const int j = lane + 64 * c;
                    d[c] = 1024;               // beyond every threshold: not counted
                    if (c < nc && j < N) {
                        const uint4 q0 = rows[2 * j], q1 = rows[2 * j + 1];
                        d[c] = __popc(r0.x ^ q0.x) + __popc(r0.y ^ q0.y) + __popc(r0.z ^ q0.z) + __popc(r0.w ^ q0.w) +
                               __popc(r1.x ^ q1.x) + __popc(r1.y ^ q1.y) + __popc(r1.z ^ q1.z) + __popc(r1.w ^ q1.w);
                    }
                }
                int lo = 0, hi = 256;
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    int cnt = 0;
#pragma unroll
                    for (int c = 0; c < MP_MAX_CHUNKS; c++)
                        if (c < nc) cnt += __popcll(__ballot(d[c] <= mid));
                    if (cnt >= need) hi = mid;
                    else lo = mid + 1;
                }
                key = min(key, (lo << 10) | i);
            }
        }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) key = min(key, __shfl_xor(key, o, 64));
        __syncthreads();                       // the last point's reads of s_key
        if (lane == 0) s_key[wv] = key;
        __syncthreads();
        const int idx = min(min(s_key[0], s_key[1]), min(s_key[2], s_key[3])) & 1023;
        if (threadIdx.x == 0) best[p] = idx;
        if (out_desc && threadIdx.x < 2)
            ((uint4*)(out_desc + (size_t)p * 32))[threadIdx.x] = rows[2 * idx + threadIdx.x];
    }
}

// max_obs: the most observations a point has.
extern "C" hipError_t orb_launch_distinctive(const uint8_t* desc, const int* offsets, int n_points, int max_obs,
                                             int* best, uint8_t* out_desc, hipStream_t st)
{
    if (n_points <= 0) return hipSuccess;
    distinctive_kernel<<<(n_points + 3) / 4, 256, 0, st>>>(desc, offsets, n_points, best, out_desc);
    if (max_obs > 64)
        distinctive_large_kernel<<<min(n_points, 2048), 256, 0, st>>>(desc, offsets, n_points, best, out_desc);
    return hipGetLastError();
}
