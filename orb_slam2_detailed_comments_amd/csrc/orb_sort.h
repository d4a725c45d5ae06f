// orb_sort.h -- bitonic sort of a workgroup's keys in registers (gfx950).
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

// The value of lane (lane ^ X) of a wavefront: DPP moves for X < 16, the LDS
// crossbar beyond.
template <int X>
__device__ __forceinline__ unsigned lane_xor(unsigned v)
{
    if constexpr (X == 1) return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
    else if constexpr (X == 2) return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4E, 0xF, 0xF, false);   // [2,3,0,1]
    else if constexpr (X == 4)                     // xor 7 (half mirror), then xor 3 (quad_perm [3,2,1,0])
        return (unsigned)__builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp((int)v, 0x141, 0xF, 0xF, false), 0x1B, 0xF, 0xF,
                                                  false);
    else if constexpr (X == 8) return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xF, 0xF, false);  // row_ror:8
    else return (unsigned)__shfl_xor((int)v, X, 64);
}

// Ascending bitonic sort of npow (a power of two, <= 1024 E) keys held E per
// thread, key i = E * tid + r, by a workgroup of 1024; keys past npow are
// larger than all others and stay.  Steps over less than E keys stay in a
// thread and steps over less than 64 E in a wavefront; only the longer ones
// (10 of the 66 for 2048 keys) go through LDS, with two barriers each.
template <int E, class K>
__device__ __forceinline__ void block_sort(K (&v)[E], int npow, K* lds)
{
    const int tid = threadIdx.x, i0 = E * tid;
    // keeps the smaller key where key i is the pair's lower place of an
    // ascending run, or the upper place of a descending one
    auto pick = [](K a, K o, bool small) { return (a < o) == small ? a : o; };
    auto lanes = [&](auto x, int k) {
        constexpr int X = decltype(x)::value;
        if (X * E >= k) return;
#pragma unroll
        for (int r = 0; r < E; r++) {
            K o = lane_xor<X>((unsigned)v[r]);
            if constexpr (sizeof(K) == 8) o |= (K)lane_xor<X>((unsigned)(v[r] >> 32)) << 32;
            v[r] = pick(v[r], o, ((i0 & (X * E)) == 0) == (((i0 + r) & k) == 0));
        }
    };
    for (int k = 2; k <= npow; k <<= 1) {
        for (int j = k >> 1; j >= 64 * E; j >>= 1) {
            __syncthreads();
#pragma unroll
            for (int r = 0; r < E; r++) lds[r * 1024 + tid] = v[r];
            __syncthreads();
            const int ot = tid ^ (j / E);
#pragma unroll
            for (int r = 0; r < E; r++) v[r] = pick(v[r], lds[r * 1024 + ot], ((i0 & j) == 0) == ((i0 & k) == 0));
        }
        lanes(std::integral_constant<int, 32>{}, k);
        lanes(std::integral_constant<int, 16>{}, k);
        lanes(std::integral_constant<int, 8>{}, k);
        lanes(std::integral_constant<int, 4>{}, k);
        lanes(std::integral_constant<int, 2>{}, k);
        lanes(std::integral_constant<int, 1>{}, k);
#pragma unroll
        for (int j = E / 2; j > 0; j >>= 1) {
            if (j >= k) continue;
#pragma unroll
            for (int r = 0; r < E; r++) {
                if (r & j) continue;
                const bool up = ((i0 + r) & k) == 0;
                const K a = v[r], b = v[r | j];
                v[r] = pick(a, b, up);
                v[r | j] = pick(b, a, !up);
            }
        }
    }
    __syncthreads();
}
