// orb_bow.hip -- gfx950 kernels for the DBoW2 vocabulary transform
// (Thirdparty/DBoW2/DBoW2/TemplatedVocabulary.h), as ORB-SLAM2 calls it from
// Frame::ComputeBoW (src/Frame.cc:704-718):
//   voc_transform_kernel  transform(feature, word_id, weight, nid, levelsup)
//                         (TemplatedVocabulary.h:1240-1290) for every row
//   voc_bow_kernel        transform(features, BowVector, FeatureVector,
//                         levelsup) (:1136-1206): per image, the word-sorted
//                         BowVector with the reference's weighting and
//                         normalisation, and the node-sorted FeatureVector
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "orb_sort.h"
#include "orb_types.h"

#define VOC_LANES 16                 // lanes per descriptor: one per child
#define BOW_CAP 4096                 // descriptors per image (LDS sort)

// Descend from the root: at each level the 16 lanes of a group take one
// child each (more than 16 children loop), key = distance << 22 | child
// index (the host admits < 2^22 children a node), and the group minimum is
// the reference's strict-< first minimum.
// Each lane loads its child's descriptor and its child's (first, count) in
// the same round, so the chosen child's children are known without another
// dependent load.
__global__ __launch_bounds__(256) void voc_transform_kernel(VocDev V, const uint8_t* __restrict__ desc, int n,
                                                            int levelsup, int* __restrict__ word_out,
                                                            double* __restrict__ weight_out, int* __restrict__ nid_out)
{
    const int sub = threadIdx.x & (VOC_LANES - 1);
    const int row = blockIdx.x * (256 / VOC_LANES) + (threadIdx.x / VOC_LANES);
    const bool live = row < n;
    const int rr = live ? row : 0;
    const uint4 q0 = *(const uint4*)(desc + (size_t)rr * 32), q1 = *(const uint4*)(desc + (size_t)rr * 32 + 16);
    const int nid_level = V.L - levelsup;
    int node = 0, nid = 0;
    int2 meta = V.meta[0];
    for (int level = 1; level <= V.max_depth && meta.y > 0; level++) {
        unsigned best = 0xFFFFFFFFu;
        int2 bmeta = make_int2(0, 0);
        for (int j = sub; j < meta.y; j += VOC_LANES) {
            const int c = meta.x + j;
            const uint4 d0 = V.desc[2 * c], d1 = V.desc[2 * c + 1];
            const int2 cm = V.meta[c];
            const unsigned d = __popc(q0.x ^ d0.x) + __popc(q0.y ^ d0.y) + __popc(q0.z ^ d0.z) +
                               __popc(q0.w ^ d0.w) + __popc(q1.x ^ d1.x) + __popc(q1.y ^ d1.y) +
                               __popc(q1.z ^ d1.z) + __popc(q1.w ^ d1.w);
            const unsigned key = (d << 22) | (unsigned)j;
            if (key < best) {
                best = key;
                bmeta = cm;
            }
        }
#pragma unroll
        for (int o = VOC_LANES / 2; o > 0; o >>= 1) {
            const unsigned ob = __shfl_xor(best, o, VOC_LANES);
            const int ox = __shfl_xor(bmeta.x, o, VOC_LANES), oy = __shfl_xor(bmeta.y, o, VOC_LANES);
            if (ob < best) {
                best = ob;
                bmeta = make_int2(ox, oy);
            }
        }
        node = meta.x + (int)(best & 0x3FFFFFu);
        meta = bmeta;
        if (level == nid_level) nid = node;
    }
    if (live && sub == 0) {
        word_out[row] = V.word_id[node];
        weight_out[row] = V.weight[node];
        if (nid_out) nid_out[row] = nid_level <= 0 ? 0 : V.orig_id[nid];
    }
}

// Exclusive scan over the 1024 threads, and the total.
__device__ __forceinline__ int block_excl_scan_1024(int x, int* sc, int* total)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int inc = x;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(inc, o, 64);
        if (lane >= o) inc += y;
    }
    if (lane == 63) sc[wv] = inc;
    __syncthreads();
    int base = 0, all = 0;
#pragma unroll
    for (int w = 0; w < 16; w++) {
        const int c = sc[w];
        base += w < wv ? c : 0;
        all += c;
    }
    *total = all;
    return base + inc - x;
}

// Two workgroups per image (1024 threads): block 2i sorts image i's rows by
// (word, feature) and writes its BowVector, block 2i + 1 sorts them by (node,
// feature) and writes its FeatureVector.  Rows with weight > 0 only (the
// reference's "not stopped" test).  BowVector: under TF / TF_IDF a word's
// value is its rows' weights added in feature order (addWeight), under IDF /
// BINARY the weight of its first row (addIfNotExist); TF / TF_IDF without
// normalisation then divide by the number of words, and normalising scorings
// divide by the L1 or L2 norm summed in word order (BowVector::normalize).
// FeatureVector: node-sorted, feature indices ascending within a node
// (addFeature in index order).
// Bound: latency of the sort's steps and of the norm's chain of additions.
// 16 images x 2000 rows: 31 us, 17 of them the norm (its terms as a chain of
// 2000 dependent additions); one workgroup per image with the sorts through
// LDS and the chain over strided reads took 85 us.
template <int E>
__device__ __forceinline__ void bow_image(const VocDev& V, const BowJob& J, int image, bool fv,
                                          const int* __restrict__ word, const double* __restrict__ wgt,
                                          const int* __restrict__ nidv, int* __restrict__ bow_word,
                                          double* __restrict__ bow_value, int* __restrict__ n_bow,
                                          int* __restrict__ fv_node, int* __restrict__ fv_feat,
                                          int* __restrict__ n_fv, unsigned long long* key, int* sc,
                                          double* s_norm)
{
    const int tid = threadIdx.x, n = min(J.n, BOW_CAP);
    const int* id = fv ? nidv : word;
    unsigned long long v[E];
    int m = 0;
#pragma unroll
    for (int r = 0; r < E; r++) {
        const int i = r * 1024 + tid;              // any order: the sort places them
        const bool live = i < n && wgt[J.off + min(i, n - 1)] > 0;
        v[r] = live ? ((unsigned long long)(unsigned)id[J.off + i] << 32) | (unsigned)i : ~0ull;
        m += __syncthreads_count(live);
    }
    int npow = 2;
    while (npow < n) npow <<= 1;
    if (npow < 1024 * E) {                         // keys r * 1024 + tid to places E tid + r, so that a short
        // list's keys lie in the first npow places
#pragma unroll
        for (int r = 0; r < E; r++) key[r * 1024 + tid] = v[r];
        __syncthreads();
#pragma unroll
        for (int r = 0; r < E; r++) v[r] = key[E * tid + r];
    }
    block_sort<E>(v, npow, key);
    if (fv) {
#pragma unroll
        for (int r = 0; r < E; r++) {
            const int i = E * tid + r;
            if (i < m) {
                fv_node[J.off + i] = (int)(unsigned)(v[r] >> 32);
                fv_feat[J.off + i] = (int)(unsigned)v[r];
            }
        }
        if (tid == 0) n_fv[image] = m;
        return;
    }
#pragma unroll
    for (int r = 0; r < E; r++) key[E * tid + r] = v[r];
    __syncthreads();
    const bool tf = V.weighting == 0 || V.weighting == 1;
    const bool must = V.scoring != 5;
    const bool l2 = V.scoring == 1;
    // heads of word runs among this thread's places, and their values
    bool head[E];
    double hv[E];
    int nh = 0;
#pragma unroll
    for (int r = 0; r < E; r++) {
        const int i = E * tid + r;
        head[r] = i < m && (i == 0 || (unsigned)(key[max(i, 1) - 1] >> 32) != (unsigned)(v[r] >> 32));
        hv[r] = head[r] ? wgt[J.off + (int)(unsigned)v[r]] : 0.0;
        nh += head[r] ? 1 : 0;
    }
    if (tf) {
#pragma unroll
        for (int r = 0; r < E; r++)
            if (head[r])
                for (int i = E * tid + r + 1; i < m && (unsigned)(key[i] >> 32) == (unsigned)(v[r] >> 32); i++)
                    hv[r] += wgt[J.off + (int)(unsigned)key[i]];
    }
    int nb;
    int rank = block_excl_scan_1024(nh, sc, &nb);  // its barrier ends the reads of key above
    // what each word adds to the norm, in word order
    double* term = reinterpret_cast<double*>(key);
    const int rank0 = rank;
#pragma unroll
    for (int r = 0; r < E; r++)
        if (head[r]) term[rank++] = l2 ? hv[r] * hv[r] : fabs(hv[r]);
    // zeros behind the last term: adding them leaves the norm as it is
    if (tid < 16 && nb + tid < 1024 * E) term[nb + tid] = 0.0;
    __syncthreads();
    if (must && tid == 0) {
        // one addition after another; the next eight terms are read while
        // eight are added
        double norm = 0.0, t[8], u[8];
#pragma unroll
        for (int q = 0; q < 8; q++) t[q] = term[q];
        for (int i = 0; i < nb; i += 16) {         // nb <= 1024 E, a multiple of 16
            const int next = min(i + 16, 1024 * E - 8);
#pragma unroll
            for (int q = 0; q < 8; q++) u[q] = term[i + 8 + q];
#pragma unroll
            for (int q = 0; q < 8; q++) norm += t[q];
#pragma unroll
            for (int q = 0; q < 8; q++) t[q] = term[next + q];
#pragma unroll
            for (int q = 0; q < 8; q++) norm += u[q];
        }
        *s_norm = l2 ? sqrt(norm) : norm;
    }
    if (tid == 0) n_bow[image] = nb;
    __syncthreads();
    const double norm = must ? *s_norm : 0.0;
    rank = rank0;
#pragma unroll
    for (int r = 0; r < E; r++)
        if (head[r]) {
            double x = hv[r];
            if (tf && !must) x = x / (double)nb;
            if (must && norm > 0.0) x = x / norm;
            bow_word[J.off + rank] = (int)(unsigned)(v[r] >> 32);
            bow_value[J.off + rank++] = x;
        }
}

__global__ __launch_bounds__(1024) void voc_bow_kernel(VocDev V, const BowJob* __restrict__ jobs,
                                                       const int* __restrict__ word, const double* __restrict__ wgt,
                                                       const int* __restrict__ nidv, int* __restrict__ bow_word,
                                                       double* __restrict__ bow_value, int* __restrict__ n_bow,
                                                       int* __restrict__ fv_node, int* __restrict__ fv_feat,
                                                       int* __restrict__ n_fv)
{
    __shared__ unsigned long long key[BOW_CAP];   // sort scratch; later the norm's terms (as double)
    __shared__ int sc[16];
    __shared__ double s_norm;
    const int image = blockIdx.x >> 1;
    const bool fv = blockIdx.x & 1;
    const BowJob J = jobs[image];
#define ORB_BOW(E) \
    bow_image<E>(V, J, image, fv, word, wgt, nidv, bow_word, bow_value, n_bow, fv_node, fv_feat, n_fv, key, sc, &s_norm)
    if (J.n <= 1024) ORB_BOW(1);
    else if (J.n <= 2048) ORB_BOW(2);
    else ORB_BOW(4);
#undef ORB_BOW
}

extern "C" hipError_t orb_launch_voc_transform(const VocDev* V, const uint8_t* desc, int n, int levelsup,
                                               int* word, double* weight, int* nid, hipStream_t st)
{
    if (n <= 0) return hipSuccess;
    const int per_block = 256 / VOC_LANES;
    voc_transform_kernel<<<(n + per_block - 1) / per_block, 256, 0, st>>>(*V, desc, n, levelsup, word, weight, nid);
    return hipGetLastError();
}

extern "C" hipError_t orb_launch_voc_bow(const VocDev* V, const BowJob* jobs, int n_images, const int* word,
                                         const double* weight, const int* nid, int* bow_word, double* bow_value,
                                         int* n_bow, int* fv_node, int* fv_feat, int* n_fv, hipStream_t st)
{
    if (n_images <= 0) return hipSuccess;
    voc_bow_kernel<<<2 * n_images, 1024, 0, st>>>(*V, jobs, word, weight, nid, bow_word, bow_value, n_bow, fv_node,
                                              fv_feat, n_fv);
    return hipGetLastError();
}
