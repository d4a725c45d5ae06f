// orb_winmatch.hip -- ORBmatcher::SearchForInitialization
// (src/ORBmatcher.cc:573-717) over the Frame keypoint grid
// (Frame::AssignFeaturesToGrid / PosInGrid / GetFeaturesInArea,
// src/Frame.cc:399-423, 590-700), for many frame pairs per call.
//
// The reference visits F1's keypoints in order, and a candidate i2 is skipped
// when an earlier match already holds it at a distance <= this one
// (vMatchedDistance), so each query depends on all earlier ones.  The work
// splits into
//   win_grid_kernel    F2's grid: keypoints sorted by (cell = ix*48 + iy,
//                      index), so the cells of one grid column ix are one
//                      contiguous run, and GetFeaturesInArea's order (ix
//                      outer, iy inner, index order within a cell) is the
//                      sorted order over the window's columns
//   win_fill_kernel    per query: the ordered (i2, distance) candidate list
//   win_round_kernel   one round of the in-order pass resolved in parallel
//                      (below), 16 lanes per query
//   win_finish_kernel  per pair: vnMatches12, nmatches, the rotation check and
//                      vbPrevMatched from the settled round's outcomes
//   win_greedy_kernel  per pair (one wavefront): the reference's sequential
//                      pass over the queries, each query's list reduced
//                      across the lanes, state (vMatchedDistance,
//                      vnMatches21, vnMatches12, the rotation histogram) in
//                      LDS; for pairs whose rounds did not settle
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "orb_sort.h"
#include "orb_types.h"

#define WIN_COLS 64
#define WIN_ROWS 48
#define WIN_CELLS (WIN_COLS * WIN_ROWS)
#define WIN_CAP 4096                 // keypoints per frame
#define WIN_PER (WIN_CAP / 1024)     // of them per thread of a workgroup of 1024
#define WIN_HISTO 30

// The cells of GetFeaturesInArea(x, y, r): columns cx0 .. cx1, rows cy0 ..
// cy1 of the grid; false if there are none.
__device__ __forceinline__ bool grid_window(float minX, float maxX, float minY, float maxY, float x, float y, float r,
                                            int* cx0, int* cx1, int* cy0, int* cy1)
{
    const float invW = static_cast<float>(WIN_COLS) / static_cast<float>(maxX - minX);
    const float invH = static_cast<float>(WIN_ROWS) / static_cast<float>(maxY - minY);
    *cx0 = max(0, (int)floorf((x - minX - r) * invW));
    *cx1 = min(WIN_COLS - 1, (int)ceilf((x - minX + r) * invW));
    *cy0 = max(0, (int)floorf((y - minY - r) * invH));
    *cy1 = min(WIN_ROWS - 1, (int)ceilf((y - minY + r) * invH));
    return *cx0 < WIN_COLS && *cx1 >= 0 && *cy0 < WIN_ROWS && *cy1 >= 0;
}

// Keypoints in the window's cells, by a group of G lanes (all of them call).
// A negative radius (negative threshold or window) can put the last row before
// the first: such columns hold none, as in the reference's loops.
template <int G>
__device__ __forceinline__ int grid_count(const int* __restrict__ cell_start, int cx0, int cx1, int cy0, int cy1)
{
    const int sub = threadIdx.x & (G - 1);
    int n = 0;
    for (int ix = cx0 + sub; ix <= cx1; ix += G)
        n += max(cell_start[ix * WIN_ROWS + cy1 + 1] - cell_start[ix * WIN_ROWS + cy0], 0);
#pragma unroll
    for (int o = 1; o < G; o <<= 1) n += __shfl_xor(n, o, G);
    return n;
}

// The window's keypoints in the reference's order (column by column; a
// column's cells are one run of rec) by a group of G lanes: a lane per column
// reads its run, and the runs of G columns are walked as one list, G entries
// at a time.  Calls f(record, position) for those that pass take(record);
// returns their number.  Branches are uniform within a group.
template <int G, class T, class F>
__device__ __forceinline__ int grid_enumerate(const int* __restrict__ cell_start, const float4* __restrict__ rec,
                                              int cx0, int cx1, int cy0, int cy1, T&& take, F&& f)
{
    const int sub = threadIdx.x & (G - 1), gbase = threadIdx.x & 63 & ~(G - 1);
    int pos = 0;
    for (int c0 = cx0; c0 <= cx1; c0 += G) {
        const int ix = c0 + sub;
        int a = 0, len = 0;
        if (ix <= cx1) {
            a = cell_start[ix * WIN_ROWS + cy0];
            len = max(cell_start[ix * WIN_ROWS + cy1 + 1] - a, 0);
        }
        int inc = len;                             // inclusive scan of the run lengths
#pragma unroll
        for (int o = 1; o < G; o <<= 1) {
            const int y = __shfl_up(inc, o, G);
            if (sub >= o) inc += y;
        }
        const int tot = __shfl(inc, G - 1, G);
        const int start = a - (inc - len);         // rec index of list entry t of this column: start + t
        for (int t0 = 0; t0 < tot; t0 += G) {
            const int t = t0 + sub;
            int col = 0;                           // first column whose scan exceeds t
#pragma unroll
            for (int o = G / 2; o > 0; o >>= 1)
                if (__shfl(inc, col + o - 1, G) <= t) col += o;
            const int j = __shfl(start, col, G) + t;
            float4 k = make_float4(0.f, 0.f, 0.f, 0.f);
            bool ok = false;
            if (t < tot) {
                k = rec[j];
                ok = take(k);
            }
            const unsigned long long all = __ballot(ok) >> gbase;
            const unsigned long long bal = G == 64 ? all : all & ((1ull << G) - 1ull);
            if (ok) f(k, pos + __popcll(bal & ((1ull << sub) - 1ull)));
            pos += __popcll(bal);
        }
    }
    return pos;
}

// Room for n list entries of each group of a workgroup of 256 (n is the same
// for a group's G lanes, 0 where there is no query): *off receives the
// group's first entry; false where the lists do not fit.  One atomic per
// workgroup, and another where the frame's region is full: the frames' regions
// keep them off one counter (25 ns an append, one after another, 1800
// workgroups in 16 frames of 1800 queries).
template <int G>
__device__ __forceinline__ bool take_entries(int n, const ListRoom& R, unsigned long long* off)
{
    __shared__ int s_n[256 / G];
    __shared__ unsigned long long s_base;
    __shared__ int s_fits;
    const int g = threadIdx.x / G;
    if ((threadIdx.x & (G - 1)) == 0) s_n[g] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        int all = 0;
        for (int i = 0; i < 256 / G; i++) all += s_n[i];
        const unsigned long long want = (unsigned)all;
        const unsigned long long o = want ? atomicAdd(R.asked, want) : 0;
        s_base = R.start + o;
        s_fits = 1;
        if (o + want > R.cap) {
            const unsigned long long os = atomicAdd(R.asked_shared, want);
            s_base = R.shared_start + os;
            s_fits = os + want <= R.shared_cap;
        }
    }
    __syncthreads();
    unsigned long long o = s_base;
    for (int i = 0; i < g; i++) o += (unsigned)s_n[i];
    *off = s_fits ? o : 0;
    return s_fits != 0;
}

// Cell of keypoint (x, y) (PosInGrid: round() of the float offset times the
// float inverse cell size), or -1 outside the grid and for keypoints that no
// query can take: for SearchForInitialization those above level 0 (minLevel =
// maxLevel = 0), for SearchByProjection those a map point with observations
// holds.
__device__ __forceinline__ int grid_cell(const WinPair& P, int i, float x, float y, int octave)
{
    const float invW = static_cast<float>(WIN_COLS) / static_cast<float>(P.maxX - P.minX);
    const float invH = static_cast<float>(WIN_ROWS) / static_cast<float>(P.maxY - P.minY);
    const int px = (int)roundf((x - P.minX) * invW), py = (int)roundf((y - P.minY) * invH);
    const bool can = P.occupied ? P.occupied[i] == 0 : octave == 0;
    return px >= 0 && px < WIN_COLS && py >= 0 && py < WIN_ROWS && can ? px * WIN_ROWS + py : -1;
}

// Place of every keypoint by sorting (cell << 20 | index); cells' first
// places by bisection.  For frames with a crowded cell.
template <int E>
__device__ __forceinline__ void grid_by_sort(const WinPair& P, int n, const int (&cell)[WIN_PER], unsigned* key,
                                             unsigned short* place)
{
    const int tid = threadIdx.x;
    unsigned v[E];
#pragma unroll
    for (int r = 0; r < E; r++) {
        const int i = r * 1024 + tid;
        v[r] = i < n ? ((unsigned)(cell[r] < 0 ? 4095 : cell[r]) << 20) | (unsigned)i : 0xFFFFFFFFu;
    }
    int npow = 2;
    while (npow < n) npow <<= 1;
    if (npow < 1024 * E) {                         // keys to places E tid + r: the first npow hold all of them
#pragma unroll
        for (int r = 0; r < E; r++) key[r * 1024 + tid] = v[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < E; r++) v[r] = key[E * tid + r];
    }
    block_sort<E>(v, npow, key);
#pragma unroll
    for (int r = 0; r < E; r++) {
        key[E * tid + r] = v[r];
        if (v[r] != 0xFFFFFFFFu) place[v[r] & 0xFFFFFu] = (unsigned short)(E * tid + r);
    }
    __syncthreads();
    for (int c = tid; c <= WIN_CELLS; c += 1024) {
        int lo = 0, hi = n;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if ((int)(key[mid] >> 20) < c) lo = mid + 1;
            else hi = mid;
        }
        P.cell_start[c] = lo;
    }
}

// One workgroup per pair: the first place of every cell and the keypoints'
// records in (cell, index) order.  A counting sort in LDS: cells counted with
// atomics, scanned, keypoints scattered in arrival order and then ranked by
// index among their cell's few; a frame with more than GRID_CROWD keypoints
// in a cell, whose ranking would grow with the square, is sorted.  Bound:
// latency of one workgroup.  2000 keypoints: 8 us (17 with the sort in
// registers, 36 with a sort through LDS).
#define GRID_CROWD 32
__global__ __launch_bounds__(1024) void win_grid_kernel(const WinPair* __restrict__ pairs)
{
    static_assert(WIN_CELLS < 4 * 1024 && WIN_CAP == WIN_PER * 1024, "four cells and keypoints a thread");
    __shared__ int start[4 * 1024];
    __shared__ unsigned key[WIN_CAP];
    __shared__ unsigned short place[WIN_CAP];
    __shared__ int part[16];
    const WinPair& P = pairs[blockIdx.x];
    const int n = P.n2, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
#pragma unroll
    for (int r = 0; r < 4; r++) start[r * 1024 + tid] = 0;
    if (P.changed) {   // SearchForInitialization's rounds: rounds 0 and 1 write claim buffers 1 and 2
        for (int i = tid; i < n; i += 1024) P.ccnt[0][i] = P.ccnt[1][i] = 0;
        for (int k = tid; k < ORB_WIN_MAXIT; k += 1024) P.changed[k] = k == 0 ? 1 : 4;   // bit 2: not run
    }
    if (tid == 0) *P.room.asked = 0;
    if (tid == 0 && blockIdx.x == 0) *P.room.asked_shared = 0;
    float4 rec[WIN_PER];
    int cell[WIN_PER], at[WIN_PER];
#pragma unroll
    for (int r = 0; r < WIN_PER; r++) {
        const int i = r * 1024 + tid;
        cell[r] = -1;
        if (i < n) {
            const OrbKeyPoint* k = P.kp2 + i;
            const float x = k->x, y = k->y;
            const int octave = k->octave;
            rec[r] = make_float4(x, y, P.uright ? P.uright[i] : 0.f, __int_as_float(i | (octave << 12)));
            cell[r] = grid_cell(P, i, x, y, octave);
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < WIN_PER; r++) at[r] = cell[r] >= 0 ? atomicAdd(&start[cell[r]], 1) : 0;
    __syncthreads();
    const int4 c4 = *(const int4*)&start[4 * tid];
    const int sum = c4.x + c4.y + c4.z + c4.w;
    int inc = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
    }
    if (lane == 63) part[wv] = inc;
    const bool crowd = __syncthreads_or(max(max(c4.x, c4.y), max(c4.z, c4.w)) > GRID_CROWD);
    if (crowd) {
        if (n <= 1024) grid_by_sort<1>(P, n, cell, key, place);
        else if (n <= 2048) grid_by_sort<2>(P, n, cell, key, place);
        else grid_by_sort<4>(P, n, cell, key, place);
#pragma unroll
        for (int r = 0; r < WIN_PER; r++)
            if (cell[r] >= 0) P.rec[place[r * 1024 + tid]] = rec[r];
        return;
    }
    int base = inc - sum;
#pragma unroll
    for (int w = 0; w < 16; w++) base += w < wv ? part[w] : 0;
    const int4 s4 = make_int4(base, base + c4.x, base + c4.x + c4.y, base + c4.x + c4.y + c4.z);
    *(int4*)&start[4 * tid] = s4;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int c = 4 * tid + e;
        if (c <= WIN_CELLS) P.cell_start[c] = e == 0 ? s4.x : (e == 1 ? s4.y : (e == 2 ? s4.z : s4.w));
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < WIN_PER; r++)
        if (cell[r] >= 0) key[start[cell[r]] + at[r]] = (unsigned)(r * 1024 + tid);
    __syncthreads();
#pragma unroll
    for (int r = 0; r < WIN_PER; r++)
        if (cell[r] >= 0) {
            const int a = start[cell[r]], b = start[cell[r] + 1];
            int rank = 0;
            for (int j = a; j < b; j++) rank += key[j] < (unsigned)(r * 1024 + tid) ? 1 : 0;
            P.rec[a + rank] = rec[r];
        }
}

__device__ __forceinline__ int row_distance(const uint4 a0, const uint4 a1, const uint8_t* b)
{
    const uint4 b0 = *(const uint4*)b, b1 = *(const uint4*)(b + 16);
    return __popc(a0.x ^ b0.x) + __popc(a0.y ^ b0.y) + __popc(a0.z ^ b0.z) + __popc(a0.w ^ b0.w) +
           __popc(a1.x ^ b1.x) + __popc(a1.y ^ b1.y) + __popc(a1.z ^ b1.z) + __popc(a1.w ^ b1.w);
}

// grid (ceil(max n1 / (256 / WIN_G)), pairs): WIN_G lanes per F1 keypoint.
// Each level-0 query takes room for all its window's keypoints and stores the
// (i2, distance) of those inside the circle, in the reference's order.
// Bound: latency (a few dependent loads per query).  2000 queries, window 100:
// 9.8 us; counting, scanning and filling in turn, a wavefront per query that
// walked its window column by column, took 44 us.
#define WIN_G 32
__global__ __launch_bounds__(256) void win_fill_kernel(const WinPair* __restrict__ pairs)
{
    const WinPair& P = pairs[blockIdx.y];
    const int q = blockIdx.x * (256 / WIN_G) + threadIdx.x / WIN_G;
    const float r = (float)P.window;
    int cx0 = 0, cx1 = -1, cy0 = 0, cy1 = -1, n = 0;
    float x = 0.f, y = 0.f;
    if (q < P.n1 && P.kp1[q].octave <= 0) {
        x = P.prev[q].x;
        y = P.prev[q].y;
        if (grid_window(P.minX, P.maxX, P.minY, P.maxY, x, y, r, &cx0, &cx1, &cy0, &cy1))
            n = grid_count<WIN_G>(P.cell_start, cx0, cx1, cy0, cy1);
    }
    unsigned long long off;
    const bool fits = take_entries<WIN_G>(n, P.room, &off);
    if (q >= P.n1) return;
    int cnt = 0;
    if (n > 0 && fits) {
        const uint4 a0 = *(const uint4*)(P.d1 + (size_t)q * 32), a1 = *(const uint4*)(P.d1 + (size_t)q * 32 + 16);
        const float rr = r * r;
        int2* out = P.cand + off;
        cnt = grid_enumerate<WIN_G>(
            P.cell_start, P.rec, cx0, cx1, cy0, cy1,
            [&](const float4& k) {
                const float distx = k.x - x, disty = k.y - y;
                return distx * distx + disty * disty < rr;
            },
            [&](const float4& k, int p) {
                const int i2 = __float_as_int(k.w) & 0xFFF;
                out[p] = make_int2(i2, row_distance(a0, a1, P.d2 + (size_t)i2 * 32));
            });
    }
    if ((threadIdx.x & (WIN_G - 1)) == 0) {
        P.cnt[q] = cnt;
        P.off[q] = off;
    }
}

// The first round k >= 1 that ran, changed no outcome and read complete
// claims (round k - 1 did not overflow its slots): its outcomes are the
// in-order pass's.  0 if there is none.
// (Every lane of the wavefront calls.)
__device__ __forceinline__ int win_settled_round(const int* chg)
{
    static_assert(ORB_WIN_MAXIT <= 64 && ORB_PROJ_MAXIT <= 64, "one round per lane");
    const int k = threadIdx.x & 63;
    const bool ok = k >= 1 && k < ORB_WIN_MAXIT && chg[k] == 0 && !(chg[k - 1] & 2);
    const unsigned long long b = __ballot(ok);
    return b ? __ffsll((long long)b) - 1 : 0;
}

// The first round k >= 1 of a SearchByProjection frame that ran and changed
// nothing, or 0.  (Every lane of the wavefront calls.)
__device__ __forceinline__ int proj_settled_round(const int* chg)
{
    const int k = threadIdx.x & 63;
    const unsigned long long b = __ballot(k >= 1 && k < ORB_PROJ_MAXIT && chg[k] == 0);
    return b ? __ffsll((long long)b) - 1 : 0;
}

// One wavefront per pair.  Query by query, in index order: lanes take the
// list positions lane, lane+64, ... (ascending), skip candidates already
// held at a distance <= theirs, and keep (first minimum as distance << 12 |
// position, second smallest distance); a butterfly merge gives the
// reference's sequential best / second.  Lane 0 applies TH_LOW, the ratio
// and the steal of a matched target; the rotation histogram counts every
// match event, as rotHist's sizes do.
__global__ __launch_bounds__(64) void win_greedy_kernel(const WinPair* __restrict__ pairs, int skip_settled)
{
    __shared__ int vmd[WIN_CAP];
    __shared__ int m21[WIN_CAP];
    __shared__ int m12[WIN_CAP];
    __shared__ signed char bin[WIN_CAP];
    __shared__ int hist[WIN_HISTO];
    __shared__ int s_n;
    const WinPair& P = pairs[blockIdx.x];
    if (skip_settled && win_settled_round(P.changed) > 0) return;
    const int lane = threadIdx.x;
    const int n1 = P.n1, n2 = P.n2;
    for (int i = lane; i < n2; i += 64) {
        vmd[i] = 0x7FFFFFFF;
        m21[i] = -1;
    }
    for (int i = lane; i < n1; i += 64) {
        m12[i] = -1;
        bin[i] = -1;
    }
    if (lane < WIN_HISTO) hist[lane] = 0;
    if (lane == 0) s_n = 0;
    __syncthreads();
    const float factor = WIN_HISTO / 360.0f;
    for (int i1 = 0; i1 < n1; i1++) {
        const int L = P.cnt[i1];
        if (L == 0 || P.kp1[i1].octave > 0) continue;
        const int2* list = P.cand + P.off[i1];
        unsigned b1 = 0xFFFFFFFFu;
        int b2 = 0x7FFFFFFF;
        for (int p = lane; p < L; p += 64) {
            const int2 c = list[p];
            if (vmd[c.x] <= c.y) continue;
            const unsigned key = ((unsigned)c.y << 12) | (unsigned)p;
            if (key < b1) {
                if (b1 != 0xFFFFFFFFu) b2 = min(b2, (int)(b1 >> 12));
                b1 = key;
            } else if (c.y < b2) {
                b2 = c.y;
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const unsigned ob1 = __shfl_xor(b1, o, 64);
            const int ob2 = __shfl_xor(b2, o, 64);
            const unsigned hi = max(b1, ob1);
            int nb2 = min(b2, ob2);
            if (hi != 0xFFFFFFFFu) nb2 = min(nb2, (int)(hi >> 12));
            b1 = min(b1, ob1);
            b2 = nb2;
        }
        if (b1 == 0xFFFFFFFFu) continue;
        const int bestDist = (int)(b1 >> 12);
        if (lane == 0 && bestDist <= 50 && (float)bestDist < (float)b2 * P.nnratio) {
            const int bestIdx2 = list[b1 & 0xFFFu].x;
            if (m21[bestIdx2] >= 0) {
                m12[m21[bestIdx2]] = -1;
                s_n--;
            }
            m12[i1] = bestIdx2;
            m21[bestIdx2] = i1;
            vmd[bestIdx2] = bestDist;
            s_n++;
            if (P.check_orientation) {
                float rot = P.kp1[i1].angle - P.kp2[bestIdx2].angle;
                if (rot < 0.0f) rot += 360.0f;
                int b = (int)roundf(rot * factor);
                if (b == WIN_HISTO) b = 0;
                bin[i1] = (signed char)b;
                hist[b]++;
            }
        }
        __syncthreads();
    }
    if (P.check_orientation) {
        // ORBmatcher::ComputeThreeMaxima (:2035-2077) on the bin sizes
        __shared__ int s_ind[3];
        if (lane == 0) {
            int max1 = 0, max2 = 0, max3 = 0, ind1 = -1, ind2 = -1, ind3 = -1;
            for (int i = 0; i < WIN_HISTO; i++) {
                const int s = hist[i];
                if (s > max1) {
                    max3 = max2;
                    max2 = max1;
                    max1 = s;
                    ind3 = ind2;
                    ind2 = ind1;
                    ind1 = i;
                } else if (s > max2) {
                    max3 = max2;
                    max2 = s;
                    ind3 = ind2;
                    ind2 = i;
                } else if (s > max3) {
                    max3 = s;
                    ind3 = i;
                }
            }
            if (max2 < 0.1f * (float)max1) {
                ind2 = -1;
                ind3 = -1;
            } else if (max3 < 0.1f * (float)max1) {
                ind3 = -1;
            }
            s_ind[0] = ind1;
            s_ind[1] = ind2;
            s_ind[2] = ind3;
        }
        __syncthreads();
        int dropped = 0;
        for (int i = lane; i < n1; i += 64) {
            const int b = bin[i];
            if (b < 0 || b == s_ind[0] || b == s_ind[1] || b == s_ind[2]) continue;
            if (m12[i] >= 0) {
                m12[i] = -1;
                dropped++;
            }
        }
        for (int o = 32; o > 0; o >>= 1) dropped += __shfl_xor(dropped, o, 64);
        if (lane == 0) s_n -= dropped;
        __syncthreads();
    }
    for (int i = lane; i < n1; i += 64) {
        const int m = m12[i];
        P.m12[i] = m;
        P.prev_out[i] = m >= 0 ? make_float2(P.kp2[m].x, P.kp2[m].y) : P.prev[i];
    }
    if (lane == 0) *P.nmatch = s_n;
}

extern "C" int orb_win_queries_per_block(void) { return 256 / WIN_G; }

extern "C" hipError_t orb_launch_win_lists(const WinPair* d_pairs, int npairs, int max_n1, hipStream_t st)
{
    if (npairs <= 0) return hipSuccess;
    win_grid_kernel<<<npairs, 1024, 0, st>>>(d_pairs);
    if (max_n1 > 0)
        win_fill_kernel<<<dim3((max_n1 + 256 / WIN_G - 1) / (256 / WIN_G), npairs), 256, 0, st>>>(d_pairs);
    return hipGetLastError();
}

// ======================================================= SearchByProjection
// Both per-frame overloads of ORBmatcher::SearchByProjection
// (src/ORBmatcher.cc:72-183 with RadiusByViewingCos :186-202, and
// :1710-1889), many frames per call.
//
// The reference visits the points in order, and a keypoint claimed by an
// earlier point that has observations is skipped by later ones, so point p's
// outcome is a function of the outcomes of points < p.  Such a sequential
// pass is the unique fixed point of "recompute every outcome against the
// claims of the previous round's outcomes": by induction, round k fixes the
// first k points, and a round that changes nothing is that fixed point.
// Conflicts are local (a few px, one or two levels), so a handful of fully
// parallel rounds replace a pass over thousands of points.  A frame that has
// not settled after ORB_PROJ_MAXIT rounds gets the sequential pass.
//   proj_prep_*        the per-point arithmetic of each overload -> ProjQuery
//   win_grid_kernel    the frame's keypoint grid (as for SearchForInitialization)
//   proj_fill_kernel   per query: (keypoint, distance, octave) of the candidates
//                      that pass the static filters (levels, circle, occupied
//                      keys, mvuRight), in GetFeaturesInArea order
//   proj_round_kernel  one claim-resolution round, 16 lanes per query
//   proj_seq_kernel    the sequential pass, for frames that did not settle
//   proj_finish_kernel per frame: key_point, nmatches, the rotation check

// The frame's round state before round 0: no claims, no round run.
__device__ __forceinline__ void proj_reset(const ProjFrame& P)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < ORB_PROJ_MAXIT) P.changed[t] = t == 0 ? 1 : 4;   // bit 2: not run
    for (int i = t; i < P.n; i += gridDim.x * 256) P.claim[0][i] = P.claim[1][i] = 0x7FFFFFFF;
}

// SearchByProjection(Frame&, vector<MapPoint*>, th) per point (:82-105):
// RadiusByViewingCos compares the float cosine with the double 0.998.
__global__ __launch_bounds__(256) void proj_prep_local_kernel(ProjFrame* __restrict__ frames,
                                                              const float* __restrict__ pts, const int* __restrict__ pt_off,
                                                              const float* __restrict__ scale, int nlevels, float th)
{
    ProjFrame& P = frames[blockIdx.y];
    const int q = blockIdx.x * 256 + threadIdx.x;
    proj_reset(P);
    if (q >= P.nq) return;
    const float* src = pts + (size_t)(pt_off[blockIdx.y] + q) * 6;   // proj_x, proj_y, proj_xr, view_cos, level, flags
    const int level = __float_as_int(src[4]), fl = __float_as_int(src[5]);
    ProjQuery Q;
    const bool valid = (fl & 1) && !(fl & 2) && level >= 0 && level < nlevels;
    float r = (double)src[3] > 0.998 ? 2.5f : 4.0f;
    if (th != 1.0f) r *= th;
    Q.x = src[0];
    Q.y = src[1];
    Q.r = valid ? r * scale[level] : 0.f;
    Q.su = src[2];
    Q.minL = level - 1;
    Q.maxL = level;
    Q.flags = (valid ? ORB_PQ_VALID : 0) | (fl & 4 ? ORB_PQ_OBS : 0);
    Q.angle = 0.f;
    P.q[q] = Q;
}

// SearchByProjection(Frame& Current, const Frame& Last, th, bMono) per point
// (:1743-1795): pinhole projection of the camera-frame point, bounds, radius
// and the level window chosen by the motion along the optical axis.
// cam per frame: fx, fy, cx, cy, mbf, mb, tlc_z.
__global__ __launch_bounds__(256) void proj_prep_last_kernel(ProjFrame* __restrict__ frames,
                                                             const float* __restrict__ pts, const int* __restrict__ pt_off,
                                                             const float* __restrict__ scale, int nlevels,
                                                             const float* __restrict__ cam, int mono, float th)
{
    ProjFrame& P = frames[blockIdx.y];
    const int q = blockIdx.x * 256 + threadIdx.x;
    proj_reset(P);
    if (q >= P.nq) return;
    const float* c = cam + (size_t)blockIdx.y * 7;
    const float fx = c[0], fy = c[1], cx = c[2], cy = c[3], mbf = c[4], mb = c[5], tlc_z = c[6];
    const bool bForward = tlc_z > mb && !mono;
    const bool bBackward = -tlc_z > mb && !mono;
    const float* src = pts + (size_t)(pt_off[blockIdx.y] + q) * 6;   // xc, yc, zc, angle, octave, flags
    const int octave = __float_as_int(src[4]), fl = __float_as_int(src[5]);
    ProjQuery Q;
    Q.flags = fl & 4 ? ORB_PQ_OBS : 0;
    Q.angle = src[3];
    Q.x = Q.y = Q.r = Q.su = 0.f;
    Q.minL = Q.maxL = -1;
    const float invzc = (float)(1.0 / (double)src[2]);
    bool valid = (fl & 1) && octave >= 0 && octave < nlevels && !(invzc < 0);
    if (valid) {
        const float u = fx * src[0] * invzc + cx;
        const float v = fy * src[1] * invzc + cy;
        valid = !(u < P.minX || u > P.maxX) && !(v < P.minY || v > P.maxY);
        Q.x = u;
        Q.y = v;
        Q.r = th * scale[octave];
        Q.su = u - mbf * invzc;
        if (bForward) {
            Q.minL = octave;
            Q.maxL = -1;
        } else if (bBackward) {
            Q.minL = 0;
            Q.maxL = octave;
        } else {
            Q.minL = octave - 1;
            Q.maxL = octave + 1;
        }
    }
    if (valid) Q.flags |= ORB_PQ_VALID;
    P.q[q] = Q;
}

// grid (ceil(max nq / 16), frames): 16 lanes per query.  Each valid query
// takes room for all its window's keypoints and stores those that pass
// GetFeaturesInArea's level rule and circle and the mvuRight check (:111-118:
// the right-image u within the radius), in the reference's order.
// Bound: latency (a few dependent loads per query).  16 frames x 1800 points,
// th 15: 28 us (counting, scanning and filling in turn 91 us); 1 frame, th 3:
// 9 us (26).
__global__ __launch_bounds__(256) void proj_fill_kernel(const ProjFrame* __restrict__ frames)
{
    const ProjFrame& P = frames[blockIdx.y];
    const int q = blockIdx.x * 16 + (threadIdx.x >> 4);
    ProjQuery Q = {};
    if (q < P.nq) Q = P.q[q];
    int cx0 = 0, cx1 = -1, cy0 = 0, cy1 = -1, n = 0;
    if ((Q.flags & ORB_PQ_VALID) &&
        grid_window(P.minX, P.maxX, P.minY, P.maxY, Q.x, Q.y, Q.r, &cx0, &cx1, &cy0, &cy1))
        n = grid_count<16>(P.cell_start, cx0, cx1, cy0, cy1);
    unsigned long long off;
    const bool fits = take_entries<16>(n, P.room, &off);
    if (q >= P.nq) return;
    int cnt = 0;
    if (n > 0 && fits) {
        const uint4 a0 = *(const uint4*)(P.qdesc + (size_t)q * 32), a1 = *(const uint4*)(P.qdesc + (size_t)q * 32 + 16);
        const bool checkLevels = (Q.minL > 0) || (Q.maxL >= 0);
        const float rr = Q.r * Q.r;
        unsigned* out = P.cand + off;
        cnt = grid_enumerate<16>(
            P.cell_start, P.rec, cx0, cx1, cy0, cy1,
            [&](const float4& k) {
                const int octave = __float_as_int(k.w) >> 12;
                if (checkLevels && !(octave >= Q.minL && (Q.maxL < 0 || octave <= Q.maxL))) return false;
                const float distx = k.x - Q.x, disty = k.y - Q.y;
                if (!(distx * distx + disty * disty < rr)) return false;
                return !(k.z > 0 && fabsf(Q.su - k.z) > Q.r);
            },
            [&](const float4& k, int p) {
                const unsigned w = (unsigned)__float_as_int(k.w), i2 = w & 0xFFFu;
                out[p] = i2 | ((unsigned)row_distance(a0, a1, P.desc + (size_t)i2 * 32) << 12) | ((w >> 12) << 21);
            });
    }
    if ((threadIdx.x & 15) == 0) {
        P.cnt[q] = cnt;
        P.off[q] = off;
    }
}

// The per-point decision over its candidate list with blocked keypoints
// removed, by `width` lanes (lanes lane0 .. lane0 + width - 1 of the
// wavefront take part; all must call).  Keys are distance << 12 | list
// position, so the smallest is the first minimum in candidate order and the
// second smallest is the reference's bestDist2 holder (the first candidate
// other than the best with that distance).  Rule 1 (:120-170): accept iff
// best <= TH_HIGH and not (same level as the second and best > ratio *
// second).  Rule 2 (:1806-1834): accept iff best <= TH_HIGH.
template <int WIDTH, class B>
__device__ __forceinline__ int proj_decide(const ProjFrame& P, int q, int sub, B&& blocked)
{
    const int L = P.cnt[q];
    const unsigned* list = P.cand + P.off[q];
    unsigned k1 = 0xFFFFFFFFu, k2 = 0xFFFFFFFFu;
    for (int p = sub; p < L; p += WIDTH) {
        const unsigned c = list[p];
        if (blocked((int)(c & 0xFFFu))) continue;
        const unsigned key = (((c >> 12) & 0x1FFu) << 12) | (unsigned)p;
        if (key < k1) {
            k2 = k1;
            k1 = key;
        } else if (key < k2) {
            k2 = key;
        }
    }
#pragma unroll
    for (int o = WIDTH / 2; o > 0; o >>= 1) {
        const unsigned o1 = __shfl_xor(k1, o, WIDTH), o2 = __shfl_xor(k2, o, WIDTH);
        const unsigned lo = min(k1, o1), hi = max(k1, o1);
        k2 = min(hi, min(k2, o2));
        k1 = lo;
    }
    if (k1 == 0xFFFFFFFFu) return -1;
    const int best = (int)(k1 >> 12);
    if (best > 100) return -1;
    const unsigned c1 = list[k1 & 0xFFFu];
    if (P.rule == 1 && k2 != 0xFFFFFFFFu) {
        const unsigned c2 = list[k2 & 0xFFFu];
        const int best2 = (int)(k2 >> 12);
        if ((c1 >> 21) == (c2 >> 21) && (float)best > P.nnratio * (float)best2) return -1;
    }
    return (int)(c1 & 0xFFFu);
}

// Round k (grid (ceil(max nq / 16), frames), 16 lanes per query): outcomes
// against the claims of round k - 1, claims of these outcomes, and the reset
// of the buffer round k + 1 will fill.  A frame settled at an earlier round
// (one that ran and changed nothing) is left alone.  A round clears bit 2 of
// its flag (set: not run).
__global__ __launch_bounds__(256) void proj_round_kernel(ProjFrame* __restrict__ frames, int k)
{
    ProjFrame& P = frames[blockIdx.y];
    const int ks = proj_settled_round(P.changed);
    if (ks > 0 && ks < k) return;                      // settled: later rounds are left alone
    if (k > 0 && blockIdx.x == 0 && threadIdx.x == 0) atomicAnd(&P.changed[k], ~4);
    const int* __restrict__ claimR = P.claim[k % 3];
    int* claimW = P.claim[(k + 1) % 3];
    int* claimC = P.claim[(k + 2) % 3];
    for (int i = blockIdx.x * 256 + threadIdx.x; i < P.n; i += gridDim.x * 256) claimC[i] = 0x7FFFFFFF;
    const int q = blockIdx.x * 16 + (threadIdx.x >> 4), sub = threadIdx.x & 15;
    const bool active = q < P.nq;
    int res = -1;
    if (active && (P.q[q].flags & ORB_PQ_VALID) && P.cnt[q] > 0)
        res = proj_decide<16>(P, q, sub, [&](int i2) { return claimR[i2] < q; });
    if (active && sub == 0) {
        P.out[k & 1][q] = res;
        if (k > 0 && P.out[(k - 1) & 1][q] != res) atomicOr(&P.changed[k], 1);
        if (res >= 0 && (P.q[q].flags & ORB_PQ_OBS)) atomicMin(&claimW[res], q);
    }
}

// The reference's sequential pass (one wavefront per frame), for frames that
// have not settled: claims in LDS, recorded as soon as a point is accepted.
// Writes round 1's outcome buffer and marks round 1 settled.
__global__ __launch_bounds__(64) void proj_seq_kernel(ProjFrame* __restrict__ frames)
{
    __shared__ int claimer[WIN_CAP];
    ProjFrame& P = frames[blockIdx.x];
    if (proj_settled_round(P.changed) > 0) return;
    for (int i = threadIdx.x; i < P.n; i += 64) claimer[i] = 0;
    __syncthreads();
    for (int q = 0; q < P.nq; q++) {
        int res = -1;
        if ((P.q[q].flags & ORB_PQ_VALID) && P.cnt[q] > 0)
            res = proj_decide<64>(P, q, threadIdx.x, [&](int i2) { return claimer[i2] != 0; });
        if (threadIdx.x == 0) {
            P.out[1][q] = res;
            if (res >= 0 && (P.q[q].flags & ORB_PQ_OBS)) claimer[res] = 1;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) P.changed[1] = 0;
}

// ORBmatcher::ComputeThreeMaxima (:2035-2077) on bin sizes.
__device__ __forceinline__ void three_maxima(const int* hist, int* ind)
{
    int max1 = 0, max2 = 0, max3 = 0, ind1 = -1, ind2 = -1, ind3 = -1;
    for (int i = 0; i < WIN_HISTO; i++) {
        const int s = hist[i];
        if (s > max1) {
            max3 = max2;
            max2 = max1;
            max1 = s;
            ind3 = ind2;
            ind2 = ind1;
            ind1 = i;
        } else if (s > max2) {
            max3 = max2;
            max2 = s;
            ind3 = ind2;
            ind2 = i;
        } else if (s > max3) {
            max3 = s;
            ind3 = i;
        }
    }
    if (max2 < 0.1f * (float)max1) {
        ind2 = -1;
        ind3 = -1;
    } else if (max3 < 0.1f * (float)max1) {
        ind3 = -1;
    }
    ind[0] = ind1;
    ind[1] = ind2;
    ind[2] = ind3;
}

// One workgroup per frame: the settled round's outcomes become pt_match;
// key_point[i] = the last point that claimed keypoint i (-1 none); rule 2
// with the rotation check builds the 30-bin histogram of the claims and sets
// key_point to -2 for the claims outside its three fullest bins
// (:1838-1886), each of which takes one off nmatches.
__global__ __launch_bounds__(1024) void proj_finish_kernel(const ProjFrame* __restrict__ frames)
{
    __shared__ int owner[WIN_CAP];
    __shared__ int hist[WIN_HISTO];
    __shared__ int s_ind[3];
    __shared__ int s_count[2];
    const ProjFrame& P = frames[blockIdx.x];
    const int kc = proj_settled_round(P.changed);
    if (kc == 0 || *P.room.asked_shared > P.room.shared_cap) return;   // more rounds, or longer lists, to come
    const int* out = P.out[kc & 1];
    for (int i = threadIdx.x; i < P.n; i += 1024) owner[i] = -1;
    if (threadIdx.x < WIN_HISTO) hist[threadIdx.x] = 0;
    if (threadIdx.x < 2) s_count[threadIdx.x] = 0;
    __syncthreads();
    const bool rot = P.rule == 2 && P.check_orientation;
    const float factor = WIN_HISTO / 360.0f;
    int nacc = 0;
    for (int q = threadIdx.x; q < P.nq; q += 1024) {
        const int m = out[q];
        P.pt_match[q] = m;
        if (m < 0) continue;
        nacc++;
        atomicMax(&owner[m], q);
        if (rot) {
            float r = P.q[q].angle - P.kp[m].angle;
            if (r < 0.0f) r += 360.0f;
            int b = (int)roundf(r * factor);
            if (b == WIN_HISTO) b = 0;
            atomicAdd(&hist[b], 1);
        }
    }
    atomicAdd(&s_count[0], nacc);
    __syncthreads();
    if (rot) {
        if (threadIdx.x == 0) three_maxima(hist, s_ind);
        __syncthreads();
        int removed = 0;
        for (int q = threadIdx.x; q < P.nq; q += 1024) {
            const int m = out[q];
            if (m < 0) continue;
            float r = P.q[q].angle - P.kp[m].angle;
            if (r < 0.0f) r += 360.0f;
            int b = (int)roundf(r * factor);
            if (b == WIN_HISTO) b = 0;
            if (b == s_ind[0] || b == s_ind[1] || b == s_ind[2]) continue;
            owner[m] = -2;          // every writer stores -2: no ordering needed
            removed++;
        }
        atomicAdd(&s_count[1], removed);
        __syncthreads();
    }
    for (int i = threadIdx.x; i < P.n; i += 1024) P.key_point[i] = owner[i];
    if (threadIdx.x == 0) *P.nmatch = s_count[0] - s_count[1];
}

extern "C" hipError_t orb_launch_proj_prep(ProjFrame* d_frames, int nframes, int max_nq, int rule, const float* d_pts,
                                           const int* d_pt_off, const float* d_scale, int nlevels, const float* d_cam,
                                           int mono, float th, hipStream_t st)
{
    if (nframes <= 0) return hipSuccess;
    const dim3 g((max(max_nq, 1) + 255) / 256, nframes);
    if (rule == 1) proj_prep_local_kernel<<<g, 256, 0, st>>>(d_frames, d_pts, d_pt_off, d_scale, nlevels, th);
    else proj_prep_last_kernel<<<g, 256, 0, st>>>(d_frames, d_pts, d_pt_off, d_scale, nlevels, d_cam, mono, th);
    return hipGetLastError();
}

extern "C" int orb_proj_queries_per_block(void) { return 256 / 16; }

// d_grid: one WinPair per frame carrying the grid fields (kp2, n2, bounds,
// uright, occupied, rec, cell_start) and the lists' room.
extern "C" hipError_t orb_launch_proj_lists(const WinPair* d_grid, const ProjFrame* d_frames, int nframes, int max_nq,
                                            hipStream_t st)
{
    if (nframes <= 0) return hipSuccess;
    win_grid_kernel<<<nframes, 1024, 0, st>>>(d_grid);
    if (max_nq > 0) proj_fill_kernel<<<dim3((max_nq + 15) / 16, nframes), 256, 0, st>>>(d_frames);
    return hipGetLastError();
}

extern "C" hipError_t orb_launch_proj_rounds(ProjFrame* d_frames, int nframes, int max_nq, int k0, int k1,
                                             hipStream_t st)
{
    if (nframes <= 0) return hipSuccess;
    for (int k = k0; k < k1; k++)
        proj_round_kernel<<<dim3((max(max_nq, 1) + 15) / 16, nframes), 256, 0, st>>>(d_frames, k);
    return hipGetLastError();
}

extern "C" hipError_t orb_launch_proj_finish(ProjFrame* d_frames, int nframes, int sequential, hipStream_t st)
{
    if (nframes <= 0) return hipSuccess;
    if (sequential) proj_seq_kernel<<<nframes, 64, 0, st>>>(d_frames);
    proj_finish_kernel<<<nframes, 1024, 0, st>>>(d_frames);
    return hipGetLastError();
}

// ============================== SearchForInitialization in parallel rounds
// The reference's pass (ORBmatcher.cc:599-665) visits the F1 keypoints in
// order; query i1 skips a candidate i2 whose vMatchedDistance is <= the
// candidate's distance, and an accepted query takes i2 (stealing it from its
// holder).  A target's successive holders have strictly decreasing
// distances, so vMatchedDistance[i2] before query i1 is the smallest distance
// of the queries < i1 accepted with target i2.  Query i1's outcome is thus a
// function of the outcomes of the queries before it, and the in-order pass
// is the unique fixed point of "recompute every outcome against the claims
// of the previous round's outcomes" (round k fixes the first k queries).
// Each target keeps up to ORB_WIN_SLOTS claims (query, distance) per round;
// a round that overflows them is not trusted as the fixed point.

// Round k (grid (ceil(max n1 / 16), pairs), 16 lanes per query): outcomes
// against the claims of round k - 1, claims of these outcomes, and the reset
// of the counts round k + 1 will fill.  A pair settled at an earlier round is
// left alone.  A round clears bit 2 of its flag (set: not run).
__global__ __launch_bounds__(256) void win_round_kernel(const WinPair* __restrict__ pairs, int k)
{
    const WinPair& P = pairs[blockIdx.y];
    const int ks = win_settled_round(P.changed);
    if (ks > 0 && ks < k) return;
    if (k > 0 && blockIdx.x == 0 && threadIdx.x == 0) atomicAnd(&P.changed[k], ~4);
    const int* __restrict__ cntR = P.ccnt[k % 3];
    const unsigned* __restrict__ claimR = P.claim[k % 3];
    int* cntW = P.ccnt[(k + 1) % 3];
    unsigned* claimW = P.claim[(k + 1) % 3];
    int* cntC = P.ccnt[(k + 2) % 3];
    for (int i = blockIdx.x * 256 + threadIdx.x; i < P.n2; i += gridDim.x * 256) cntC[i] = 0;
    const int q = blockIdx.x * 16 + (threadIdx.x >> 4), sub = threadIdx.x & 15;
    const bool active = q < P.n1;
    int res = -1;
    if (active && P.cnt[q] > 0 && P.kp1[q].octave == 0) {   // the 16 lanes of a query agree
        const int L = P.cnt[q];
        const int2* list = P.cand + P.off[q];
        unsigned b1 = 0xFFFFFFFFu;
        int b2 = 0x7FFFFFFF;
        for (int p = sub; p < L; p += 16) {
            const int2 c = list[p];
            const int nc = min(cntR[c.x], ORB_WIN_SLOTS);
            bool blocked = false;
            for (int j = 0; j < nc; j++) {
                const unsigned e = claimR[(size_t)c.x * ORB_WIN_SLOTS + j];
                blocked |= (int)(e >> 9) < q && (int)(e & 511u) <= c.y;
            }
            if (blocked) continue;
            const unsigned key = ((unsigned)c.y << 12) | (unsigned)p;
            if (key < b1) {
                if (b1 != 0xFFFFFFFFu) b2 = min(b2, (int)(b1 >> 12));
                b1 = key;
            } else if (c.y < b2) {
                b2 = c.y;
            }
        }
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) {
            const unsigned ob1 = __shfl_xor(b1, o, 16);
            const int ob2 = __shfl_xor(b2, o, 16);
            const unsigned hi = max(b1, ob1);
            int nb2 = min(b2, ob2);
            if (hi != 0xFFFFFFFFu) nb2 = min(nb2, (int)(hi >> 12));
            b1 = min(b1, ob1);
            b2 = nb2;
        }
        if (b1 != 0xFFFFFFFFu) {
            const int bestDist = (int)(b1 >> 12);
            if (bestDist <= 50 && (float)bestDist < (float)b2 * P.nnratio) res = (list[b1 & 0xFFFu].x << 9) | bestDist;
        }
    }
    if (active && sub == 0) {
        P.out[k & 1][q] = res;
        if (k > 0 && P.out[(k - 1) & 1][q] != res) atomicOr(&P.changed[k], 1);
        if (res >= 0) {
            const int t = res >> 9;
            const int slot = atomicAdd(&cntW[t], 1);
            if (slot < ORB_WIN_SLOTS) claimW[(size_t)t * ORB_WIN_SLOTS + slot] = ((unsigned)q << 9) | (unsigned)(res & 511);
            else atomicOr(&P.changed[k], 2);
        }
    }
}

// One workgroup per settled pair: every accepted query is a match event (a
// rotHist entry); a target stays with its last holder (vnMatches12 of the
// others was reset by the steal); the rotation check drops the matches whose
// event lies outside the three fullest bins (:667-690); vbPrevMatched takes
// the kept matches' F2 positions (:693-695).
__global__ __launch_bounds__(1024) void win_finish_kernel(const WinPair* __restrict__ pairs)
{
    __shared__ int owner[WIN_CAP];
    __shared__ int hist[WIN_HISTO];
    __shared__ int s_ind[3];
    __shared__ int s_n;
    const WinPair& P = pairs[blockIdx.x];
    const int ks = win_settled_round(P.changed);
    if (ks == 0 || *P.room.asked_shared > P.room.shared_cap) return;   // more rounds, the sequential pass or longer lists to come
    const int* out = P.out[ks & 1];
    const int n1 = P.n1, t = threadIdx.x;
    constexpr int PER = WIN_PER;                   // queries t, t + 1024, ... of a thread, read together
    int r[PER];
    float2 pos[PER];
    float a1[PER];
#pragma unroll
    for (int e = 0; e < PER; e++) {
        const int q = t + 1024 * e;
        r[e] = -1;
        if (q < n1) {
            r[e] = out[q];
            pos[e] = P.prev[q];
            a1[e] = P.kp1[q].angle;
        }
    }
    for (int i = t; i < P.n2; i += 1024) owner[i] = -1;
    if (t < WIN_HISTO) hist[t] = 0;
    if (t == 0) s_n = 0;
    __syncthreads();
    const float factor = WIN_HISTO / 360.0f;
    int bin[PER];
    float2 at[PER];
#pragma unroll
    for (int e = 0; e < PER; e++) {
        bin[e] = -1;
        if (r[e] >= 0) {
            const int tg = r[e] >> 9;
            atomicMax(&owner[tg], t + 1024 * e);
            at[e] = make_float2(P.kp2[tg].x, P.kp2[tg].y);
            if (P.check_orientation) {
                float rot = a1[e] - P.kp2[tg].angle;
                if (rot < 0.0f) rot += 360.0f;
                int b = (int)roundf(rot * factor);
                if (b == WIN_HISTO) b = 0;
                bin[e] = b;
                atomicAdd(&hist[b], 1);
            }
        }
    }
    __syncthreads();
    if (P.check_orientation) {
        if (t == 0) three_maxima(hist, s_ind);
        __syncthreads();
    }
    int kept = 0;
#pragma unroll
    for (int e = 0; e < PER; e++) {
        const int q = t + 1024 * e;
        if (q >= n1) continue;
        const int b = bin[e];
        const bool drop = b >= 0 && b != s_ind[0] && b != s_ind[1] && b != s_ind[2];
        const bool keep = r[e] >= 0 && owner[max(r[e], 0) >> 9] == q && !drop;
        kept += keep ? 1 : 0;
        P.m12[q] = keep ? r[e] >> 9 : -1;
        P.prev_out[q] = keep ? at[e] : pos[e];
    }
    atomicAdd(&s_n, kept);
    __syncthreads();
    if (t == 0) *P.nmatch = s_n;
}

extern "C" hipError_t orb_launch_win_rounds(const WinPair* d_pairs, int npairs, int max_n1, int k0, int k1,
                                            hipStream_t st)
{
    if (npairs <= 0) return hipSuccess;
    for (int k = k0; k < k1; k++)
        win_round_kernel<<<dim3((max(max_n1, 1) + 15) / 16, npairs), 256, 0, st>>>(d_pairs, k);
    return hipGetLastError();
}

extern "C" hipError_t orb_launch_win_finish(const WinPair* d_pairs, int npairs, int sequential, hipStream_t st)
{
    if (npairs <= 0) return hipSuccess;
    win_finish_kernel<<<npairs, 1024, 0, st>>>(d_pairs);
    if (sequential) win_greedy_kernel<<<npairs, 64, 0, st>>>(d_pairs, 1);
    return hipGetLastError();
}
