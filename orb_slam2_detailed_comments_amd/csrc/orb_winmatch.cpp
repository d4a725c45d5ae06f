// orb_winmatch.cpp -- C ABI of ORBmatcher::SearchForInitialization over the
// Frame keypoint grid, for many frame pairs per call (kernels in
// orb_winmatch.hip).  A call copies its inputs to the device once, launches
// the grid, the candidate lists, four rounds and the finish, copies every
// result back and waits once; it goes on only if some pair has not settled,
// or if the lists did not fit their buffer (which then grows, so that an equal
// call fits).  Device and
// pinned buffers are the context's, grown on demand and kept between calls.
#include <chrono>
#include <cstring>
#include <vector>

#include "orb_internal.h"

using namespace orb_detail;

extern "C" int orb_win_queries_per_block(void);
extern "C" hipError_t orb_launch_win_lists(const WinPair* d_pairs, int npairs, int max_n1, hipStream_t st);
extern "C" hipError_t orb_launch_win_rounds(const WinPair* d_pairs, int npairs, int max_n1, int k0, int k1,
                                            hipStream_t st);
extern "C" hipError_t orb_launch_win_finish(const WinPair* d_pairs, int npairs, int sequential, hipStream_t st);

// Bytes to allocate where `bytes` no longer fit into `have`: the first time what
// is asked for, then a quarter more, at least 64 KB and at most 1 MB, so that a
// camera's frames, which differ by some keypoints, grow the buffers a few times
// and not with every largest frame so far (a pinned buffer costs 150-250 us).
// 60 frames of 1000, 1015, ... points: 148 us a call on average, 374 with exact
// sizes.
extern "C" size_t orb_win_capacity(size_t have, size_t bytes)
{
    if (have == 0) return bytes;
    const size_t more = std::min(std::max(bytes / 4, (size_t)64 << 10), (size_t)1 << 20);
    return (bytes + more + 4095) / 4096 * 4096;
}

namespace {

size_t up(size_t v) { return (v + 255) / 256 * 256; }

int reserve(orb_context* ctx, void** p, size_t* cap, size_t bytes)
{
    return bytes <= *cap ? ORB_OK : ctx->grow(p, cap, orb_win_capacity(*cap, bytes));
}

int reserve_pinned(orb_context* ctx, void** p, size_t* cap, size_t bytes)
{
    return bytes <= *cap ? ORB_OK : ctx->grow_pinned(p, cap, orb_win_capacity(*cap, bytes));
}

// A call's device block: what is copied in, what is copied out, then scratch.
// The outputs are packed in pinned memory at their device offsets, so that one
// copy takes them; so are the inputs (Upload).
struct Block {
    size_t in = 0, out = 0, scratch = 0;
    size_t add_in(size_t bytes) { return add(in, bytes); }
    size_t add_out(size_t bytes) { return add(out, bytes); }
    size_t add_scratch(size_t bytes) { return add(scratch, bytes); }
    static size_t add(size_t& end, size_t bytes)
    {
        const size_t o = end;
        end += up(bytes);
        return o;
    }
};

// A call's inputs on their way to the device: arrays of the caller's at the
// offsets below `tables`, then what the host keeps for the call (jobs, offsets,
// parameters) up to `in`.  Up to kWindow bytes of arrays are packed in front of
// the tables in pinned memory, and one copy takes both.  More of them go through
// the window's halves in turn, one being filled while the other is copied, and
// the tables follow: so the pinned buffer does not grow with them, whose first
// allocation costs 0.3 ms a megabyte.
// Last-frame searches of 256 frames (61 MB): first call of a context 27 ms with
// everything pinned and 8.6 so, later ones 4.37 and 3.4; 64 frames (15 MB) 7.9
// and 5.3, later 0.87 and 0.84.  Windows of 4 MB: 32 frames (7.6 MB) 525 us, 497
// in one copy; of 2 MB: 16 frames (3.8 MB) 326 us, 286 in one copy.
constexpr size_t kWindow = (size_t)8 << 20;

struct Upload {
    orb_context* ctx;
    char* d;
    char* h = nullptr;
    size_t tables, in, window;
    int half = 0;
    bool busy[2] = {false, false}, sent = false;

    Upload(orb_context* c, size_t tables_at, size_t in_bytes)
        : ctx(c), d((char*)c->d_win), tables(tables_at), in(in_bytes), window(std::min(tables_at, kWindow))
    {
    }
    Upload(const Upload&) = delete;
    Upload& operator=(const Upload&) = delete;
    // A call that ends before its tables are sent (no room for the lists) leaves
    // no copy from the window under way: the next call refills or frees it.
    ~Upload()
    {
        if (!sent && (busy[0] || busy[1])) (void)hipStreamSynchronize(ctx->stream);
    }
    size_t pinned_bytes() const { return window + (in - tables); }
    bool whole() const { return window == tables; }
    template <class T>
    T* table(size_t at) const
    {
        return (T*)(h + window + (at - tables));
    }
    int put(size_t at, const void* src, size_t bytes)
    {
        if (whole()) {
            std::memcpy(h + at, src, bytes);
            return ORB_OK;
        }
        for (size_t o = 0; o < bytes; o += kWindow / 2, half ^= 1) {
            const size_t n = std::min(bytes - o, kWindow / 2);
            char* to = h + half * (kWindow / 2);
            hipEvent_t& ev = ctx->win_ev[half];
            if (!ev) HIP_TRY(hipEventCreateWithFlags(&ev, hipEventDisableTiming));
            if (busy[half]) HIP_TRY(hipEventSynchronize(ev));
            std::memcpy(to, (const char*)src + o, n);
            HIP_TRY(hipMemcpyAsync(d + at + o, to, n, hipMemcpyHostToDevice, ctx->stream));
            HIP_TRY(hipEventRecord(ev, ctx->stream));
            busy[half] = true;
        }
        return ORB_OK;
    }
    int finish()
    {
        const size_t from = whole() ? 0 : tables;
        HIP_TRY(hipMemcpyAsync(d + from, whole() ? h : h + window, in - from, hipMemcpyHostToDevice, ctx->stream));
        sent = true;
        return ORB_OK;
    }
};

// The candidate lists' places in the context's buffer.  A pair's (or frame's)
// queries have a region of kListRegion entries each (a window holds no more
// than the frame's keypoints); workgroups past their region's end take from the
// rest of the buffer, which all share.  The regions follow from the call alone,
// so what an equal call takes from the rest is known up to the workgroups that
// straddle the regions' ends: a call that did not fit makes the buffer that
// large, and a quarter more for the next frames.
// A local-map search of 4000 keypoints, th 5 (75 entries a query): 288 us; 334
// with even shares of a buffer as large as the asked total, which the asked
// list outgrew by the shares' rounding, so that every call ran twice.
constexpr size_t kListRegion = 64;

struct Lists {
    std::vector<size_t> nq, nk;             // queries, keypoints a window can hold
    size_t regions = 0;                     // entries of all regions

    void add(int n_queries, int n_keys)
    {
        nq.push_back((size_t)n_queries);
        nk.push_back((size_t)n_keys);
        regions += region(nq.size() - 1);
    }
    size_t region(size_t i) const { return nq[i] * std::min(kListRegion, nk[i]); }

    // Entries an equal call needs, from what this one asked for; a workgroup
    // has per_block queries.
    size_t need(const unsigned long long* asked, size_t per_block) const
    {
        size_t shared = 0;
        for (size_t i = 0; i < nq.size(); i++)
            if (asked[i] > region(i)) shared += (size_t)asked[i] - region(i) + per_block * nk[i];
        return regions + shared + shared / 4;
    }

    // Room i in a buffer of `have` entries; counters: a frame's each, then the shared one.
    ListRoom room(size_t i, size_t start, size_t have, unsigned long long* counters) const
    {
        return ListRoom{counters + i, counters + nq.size(), start, region(i), regions, have - regions};
    }
};

// steps > 0: after the call's own run, `steps` more runs of the device work
// with the inputs resident in HBM, their
// mean wall time in *ms; the results returned are the call's.
int sfi_impl(orb_context* ctx, int n_pairs, const orb_keypoint* kp1, const uint8_t* desc1, const int32_t* off1,
             const orb_keypoint* kp2, const uint8_t* desc2, const int32_t* off2, const float* bounds,
             float* prev_matched, int window_size, float nn_ratio, int check_orientation, int32_t* matches12,
             int32_t* nmatches, int steps, float* ms)
{
    if (!ctx || n_pairs < 0 || (n_pairs && (!off1 || !off2 || !bounds || !matches12 || !nmatches))) return ORB_E_ARG;
    if (n_pairs == 0) return ORB_OK;
    const int N1 = off1[n_pairs], N2 = off2[n_pairs];
    if ((N1 && (!kp1 || !desc1 || !prev_matched)) || (N2 && (!kp2 || !desc2))) return ORB_E_ARG;
    int max_n1 = 0;
    for (int p = 0; p < n_pairs; p++) {
        const int a = off1[p + 1] - off1[p], b = off2[p + 1] - off2[p];
        if (a < 0 || b < 0 || off1[p] < 0 || off2[p] < 0) return ORB_E_ARG;
        if (a > 4096 || b > 4096) return ORB_E_CAPACITY;
        if (!(bounds[4 * p + 1] > bounds[4 * p]) || !(bounds[4 * p + 3] > bounds[4 * p + 2])) return ORB_E_ARG;
        max_n1 = std::max(max_n1, a);
    }
    HIP_TRY(hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    static_assert(sizeof(orb_keypoint) == sizeof(OrbKeyPoint), "keypoint layout");
    const size_t P = (size_t)n_pairs, n1 = (size_t)N1, n2 = (size_t)N2;
    Block B;
    const size_t i_kp1 = B.add_in(n1 * sizeof(OrbKeyPoint)), i_d1 = B.add_in(n1 * 32), i_prev = B.add_in(n1 * 8);
    const size_t i_kp2 = B.add_in(n2 * sizeof(OrbKeyPoint)), i_d2 = B.add_in(n2 * 32);
    const size_t i_pairs = B.add_in(P * sizeof(WinPair));
    const size_t o_m12 = B.add_out(n1 * 4), o_prev = B.add_out(n1 * 8), o_nm = B.add_out(P * 4);
    const size_t o_tot = B.add_out((P + 1) * 8), o_chg = B.add_out(P * ORB_WIN_MAXIT * 4);
    const size_t s_rec = B.add_scratch(n2 * 16), s_cells = B.add_scratch(P * (64 * 48 + 1) * 4);
    const size_t s_cnt = B.add_scratch(n1 * 4), s_off = B.add_scratch(n1 * 8);
    // round state: outcomes by parity, claims and claim counts by round mod 3
    const size_t s_out = B.add_scratch(2 * n1 * 4), s_claim = B.add_scratch(3 * n2 * ORB_WIN_SLOTS * 4);
    const size_t s_ccnt = B.add_scratch(3 * n2 * 4);
    int rc = reserve(ctx, &ctx->d_win, &ctx->win_cap, B.in + B.out + B.scratch);
    if (rc) return rc;
    Upload up_in(ctx, i_pairs, B.in);
    rc = reserve_pinned(ctx, &ctx->h_win, &ctx->hwin_cap, up_in.pinned_bytes() + B.out);
    if (rc) return rc;
    char *d_in = (char*)ctx->d_win, *d_out = d_in + B.in, *d_s = d_out + B.out;
    char* h_out = (char*)ctx->h_win + up_in.pinned_bytes();
    up_in.h = (char*)ctx->h_win;
    if (N1) {
        rc = up_in.put(i_kp1, kp1, n1 * sizeof(OrbKeyPoint));
        if (!rc) rc = up_in.put(i_d1, desc1, n1 * 32);
        if (!rc) rc = up_in.put(i_prev, prev_matched, n1 * 8);
    }
    if (N2) {
        if (!rc) rc = up_in.put(i_kp2, kp2, n2 * sizeof(OrbKeyPoint));
        if (!rc) rc = up_in.put(i_d2, desc2, n2 * 32);
    }
    if (rc) return rc;
    WinPair* pairs = up_in.table<WinPair>(i_pairs);
    Lists lists;
    for (int p = 0; p < n_pairs; p++) {
        WinPair& w = pairs[p];
        std::memset(&w, 0, sizeof(w));
        w.kp1 = (const OrbKeyPoint*)(d_in + i_kp1) + off1[p];
        w.d1 = (const uint8_t*)(d_in + i_d1) + (size_t)off1[p] * 32;
        w.kp2 = (const OrbKeyPoint*)(d_in + i_kp2) + off2[p];
        w.d2 = (const uint8_t*)(d_in + i_d2) + (size_t)off2[p] * 32;
        w.n1 = off1[p + 1] - off1[p];
        w.n2 = off2[p + 1] - off2[p];
        w.minX = bounds[4 * p];
        w.maxX = bounds[4 * p + 1];
        w.minY = bounds[4 * p + 2];
        w.maxY = bounds[4 * p + 3];
        w.prev = (const float2*)(d_in + i_prev) + off1[p];
        w.window = window_size;
        w.nnratio = nn_ratio;
        w.check_orientation = check_orientation ? 1 : 0;
        w.rec = (float4*)(d_s + s_rec) + off2[p];
        w.cell_start = (int*)(d_s + s_cells) + (size_t)p * (64 * 48 + 1);
        w.cnt = (int*)(d_s + s_cnt) + off1[p];
        w.off = (unsigned long long*)(d_s + s_off) + off1[p];
        w.m12 = (int*)(d_out + o_m12) + off1[p];
        w.prev_out = (float2*)(d_out + o_prev) + off1[p];
        w.nmatch = (int*)(d_out + o_nm) + p;
        for (int b = 0; b < 2; b++) w.out[b] = (int*)(d_s + s_out) + b * n1 + off1[p];
        for (int b = 0; b < 3; b++) {
            w.claim[b] = (unsigned*)(d_s + s_claim) + (b * n2 + off2[p]) * ORB_WIN_SLOTS;
            w.ccnt[b] = (int*)(d_s + s_ccnt) + b * n2 + off2[p];
        }
        w.changed = (int*)(d_out + o_chg) + (size_t)p * ORB_WIN_MAXIT;
        lists.add(w.n1, w.n2);
    }
    const unsigned long long* tot = (const unsigned long long*)(h_out + o_tot);
    const int* chg = (const int*)(h_out + o_chg);
    // a buffer of at least n entries, and the lists' places in it
    auto place_lists = [&](size_t n) -> int {
        const int rg = reserve(ctx, &ctx->d_wcand, &ctx->wcand_cap, std::max<size_t>(n, 1) * sizeof(int2));
        if (rg) return rg;
        size_t start = 0;
        for (int p = 0; p < n_pairs; p++) {
            pairs[p].cand = (int2*)ctx->d_wcand;
            pairs[p].room = lists.room(p, start, ctx->wcand_cap / sizeof(int2), (unsigned long long*)(d_out + o_tot));
            start += lists.region(p);
        }
        return ORB_OK;
    };
    rc = place_lists(lists.regions);
    if (!rc) rc = up_in.finish();
    if (rc) return rc;
    const WinPair* d_pairs = (const WinPair*)(d_in + i_pairs);
    auto run_device = [&]() -> int {
        const int limit = std::min(ctx->round_limit, ORB_WIN_MAXIT);
        int k = 0;
        bool settled = false;
        ctx->last_restarts = 0;
        HIP_TRY(orb_launch_win_lists(d_pairs, n_pairs, max_n1, st));
        // Rounds in chunks of 4, each followed by the finish of the pairs
        // that have settled; pairs still changing at the limit get the
        // sequential pass.
        for (;;) {
            const int k1 = std::min(limit, k + 4);
            HIP_TRY(orb_launch_win_rounds(d_pairs, n_pairs, max_n1, k, k1, st));
            k = k1;
            HIP_TRY(orb_launch_win_finish(d_pairs, n_pairs, 0, st));
            HIP_TRY(hipMemcpyAsync(h_out, d_out, B.out, hipMemcpyDeviceToHost, st));
            HIP_TRY(hipStreamSynchronize(st));
            if (tot[P] > pairs[0].room.shared_cap) {   // longer lists, from the start
                ctx->last_restarts++;
                const int rl = place_lists(lists.need(tot, orb_win_queries_per_block()));
                if (rl) return rl;
                HIP_TRY(hipMemcpyAsync(d_in + i_pairs, pairs, P * sizeof(WinPair), hipMemcpyHostToDevice, st));
                HIP_TRY(orb_launch_win_lists(d_pairs, n_pairs, max_n1, st));
                k = 0;
                continue;
            }
            settled = true;
            for (int p = 0; p < n_pairs && settled; p++) {
                const int* c = chg + (size_t)p * ORB_WIN_MAXIT;
                bool sp = false;
                for (int r = 1; r < k && !sp; r++) sp = c[r] == 0 && !(c[r - 1] & 2);
                settled = sp;
            }
            if (settled || k >= limit) break;
        }
        ctx->last_rounds = k;
        ctx->last_sequential = settled ? 0 : 1;
        if (!settled) {
            HIP_TRY(orb_launch_win_finish(d_pairs, n_pairs, 1, st));
            HIP_TRY(hipMemcpyAsync(h_out, d_out, B.out, hipMemcpyDeviceToHost, st));
            HIP_TRY(hipStreamSynchronize(st));
        }
        return ORB_OK;
    };
    rc = run_device();
    if (rc) return rc;
    if (steps > 0) {
        const auto t0 = std::chrono::steady_clock::now();
        for (int i = 0; i < steps; i++) {
            rc = run_device();
            if (rc) return rc;
        }
        *ms = (float)(std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count() / steps);
    }
    // (rows before the first pair's are not the call's to write)
    const size_t r1 = (size_t)off1[0];
    if (n1 > r1) {
        std::memcpy(matches12 + r1, h_out + o_m12 + r1 * 4, (n1 - r1) * 4);
        std::memcpy(prev_matched + 2 * r1, h_out + o_prev + r1 * 8, (n1 - r1) * 8);
    }
    std::memcpy(nmatches, h_out + o_nm, P * 4);
    return ORB_OK;
}

}  // namespace

extern "C" {

int orb_search_for_initialization(orb_context* ctx, int n_pairs, const orb_keypoint* kp1, const uint8_t* desc1,
                                  const int32_t* off1, const orb_keypoint* kp2, const uint8_t* desc2,
                                  const int32_t* off2, const float* bounds, float* prev_matched, int window_size,
                                  float nn_ratio, int check_orientation, int32_t* matches12, int32_t* nmatches)
{
    return sfi_impl(ctx, n_pairs, kp1, desc1, off1, kp2, desc2, off2, bounds, prev_matched, window_size, nn_ratio,
                    check_orientation, matches12, nmatches, 0, nullptr);
}

int orb_search_for_initialization_time(orb_context* ctx, int n_pairs, const orb_keypoint* kp1, const uint8_t* desc1,
                                       const int32_t* off1, const orb_keypoint* kp2, const uint8_t* desc2,
                                       const int32_t* off2, const float* bounds, float* prev_matched, int window_size,
                                       float nn_ratio, int check_orientation, int32_t* matches12, int32_t* nmatches,
                                       int steps, float* ms)
{
    if (steps <= 0 || !ms) return ORB_E_ARG;
    return sfi_impl(ctx, n_pairs, kp1, desc1, off1, kp2, desc2, off2, bounds, prev_matched, window_size, nn_ratio,
                    check_orientation, matches12, nmatches, steps, ms);
}

}  // extern "C"

// ---------------------------------------------------------- SearchByProjection
extern "C" hipError_t orb_launch_proj_prep(ProjFrame* d_frames, int nframes, int max_nq, int rule, const float* d_pts,
                                           const int* d_pt_off, const float* d_scale, int nlevels, const float* d_cam,
                                           int mono, float th, hipStream_t st);
extern "C" int orb_proj_queries_per_block(void);
extern "C" hipError_t orb_launch_proj_lists(const WinPair* d_grid, const ProjFrame* d_frames, int nframes, int max_nq,
                                            hipStream_t st);
extern "C" hipError_t orb_launch_proj_rounds(ProjFrame* d_frames, int nframes, int max_nq, int k0, int k1,
                                             hipStream_t st);
extern "C" hipError_t orb_launch_proj_finish(ProjFrame* d_frames, int nframes, int sequential, hipStream_t st);

namespace {

// Both overloads: rule 1 = SearchByProjection(F, vpMapPoints, th), rule 2 =
// SearchByProjection(Current, Last, th, bMono).  Point records are 24 bytes
// (orb_proj_point / orb_last_point).  Rounds run in chunks of 4 between
// reads of the per-round change flags; frames still changing after
// ORB_PROJ_MAXIT rounds get the sequential pass.
int proj_search(orb_context* ctx, int rule, int n_frames, const orb_keypoint* kp, const uint8_t* desc,
                const float* uright, const uint8_t* occupied, const int32_t* key_off, const float* bounds,
                const float* scale, int nlevels, const void* pts, const uint8_t* pdesc, const int32_t* pt_off,
                const float* cam, int mono, float th, float nnratio, int check_orientation, int32_t* pt_match,
                int32_t* key_point, int32_t* nmatches, int steps, float* ms)
{
    static_assert(sizeof(orb_proj_point) == 24 && sizeof(orb_last_point) == 24, "point records");
    if (!ctx || n_frames < 0 || nlevels < 1 || nlevels > ORB_MAX_LEVELS ||
        (n_frames && (!key_off || !pt_off || !bounds || !scale || !nmatches || (rule == 2 && !cam))))
        return ORB_E_ARG;
    if (n_frames == 0) return ORB_OK;
    const int N = key_off[n_frames], Q = pt_off[n_frames];
    if ((N && (!kp || !desc || !uright || !occupied || !key_point)) || (Q && (!pts || !pdesc || !pt_match)))
        return ORB_E_ARG;
    int max_nq = 0;
    for (int f = 0; f < n_frames; f++) {
        const int n = key_off[f + 1] - key_off[f], nq = pt_off[f + 1] - pt_off[f];
        if (n < 0 || nq < 0 || key_off[f] < 0 || pt_off[f] < 0) return ORB_E_ARG;
        if (n > 4096 || nq > (1 << 20)) return ORB_E_CAPACITY;
        if (!(bounds[4 * f + 1] > bounds[4 * f]) || !(bounds[4 * f + 3] > bounds[4 * f + 2])) return ORB_E_ARG;
        max_nq = std::max(max_nq, nq);
    }
    for (int i = 0; i < N; i++)
        if (kp[i].octave < 0 || kp[i].octave >= ORB_MAX_LEVELS) return ORB_E_ARG;
    // The rotation check bins (last angle - current angle) mod 360; keypoint
    // angles lie in [0, 360] (the reference asserts a bin in range, :1836).
    if (rule == 2 && check_orientation) {
        for (int i = 0; i < N; i++)
            if (!(kp[i].angle >= 0.f && kp[i].angle <= 360.f)) return ORB_E_ARG;
        const orb_last_point* lp = (const orb_last_point*)pts;
        for (int q = 0; q < Q; q++)
            if ((lp[q].flags & 1) && !(lp[q].angle >= 0.f && lp[q].angle <= 360.f)) return ORB_E_ARG;
    }
    HIP_TRY(hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    static_assert(sizeof(orb_keypoint) == sizeof(OrbKeyPoint), "keypoint layout");
    const size_t F = (size_t)n_frames, nk = (size_t)N, np = (size_t)Q;
    Block B;
    const size_t i_kp = B.add_in(nk * sizeof(OrbKeyPoint)), i_desc = B.add_in(nk * 32), i_ur = B.add_in(nk * 4),
                 i_occ = B.add_in(nk), i_pts = B.add_in(np * 24), i_pdesc = B.add_in(np * 32),
                 i_ptoff = B.add_in((F + 1) * 4), i_scale = B.add_in(ORB_MAX_LEVELS * 4), i_cam = B.add_in(F * 7 * 4),
                 i_grid = B.add_in(F * sizeof(WinPair)), i_frames = B.add_in(F * sizeof(ProjFrame));
    const size_t o_ptm = B.add_out(np * 4), o_keyp = B.add_out(nk * 4), o_nm = B.add_out(F * 4),
                 o_tot = B.add_out((F + 1) * 8), o_chg = B.add_out(F * ORB_PROJ_MAXIT * 4);
    const size_t s_rec = B.add_scratch(nk * 16), s_cells = B.add_scratch(F * (64 * 48 + 1) * 4),
                 s_q = B.add_scratch(np * sizeof(ProjQuery)), s_cnt = B.add_scratch(np * 4),
                 s_off = B.add_scratch(np * 8), s_out = B.add_scratch(2 * np * 4), s_claim = B.add_scratch(3 * nk * 4);
    int rc = reserve(ctx, &ctx->d_win, &ctx->win_cap, B.in + B.out + B.scratch);
    if (rc) return rc;
    Upload up_in(ctx, i_ptoff, B.in);
    rc = reserve_pinned(ctx, &ctx->h_win, &ctx->hwin_cap, up_in.pinned_bytes() + B.out);
    if (rc) return rc;
    char *d_in = (char*)ctx->d_win, *d_out = d_in + B.in, *d_s = d_out + B.out;
    char* h_out = (char*)ctx->h_win + up_in.pinned_bytes();
    up_in.h = (char*)ctx->h_win;
    if (N) {
        rc = up_in.put(i_kp, kp, nk * sizeof(OrbKeyPoint));
        if (!rc) rc = up_in.put(i_desc, desc, nk * 32);
        if (!rc) rc = up_in.put(i_ur, uright, nk * 4);
        if (!rc) rc = up_in.put(i_occ, occupied, nk);
    }
    if (Q) {
        if (!rc) rc = up_in.put(i_pts, pts, np * 24);
        if (!rc) rc = up_in.put(i_pdesc, pdesc, np * 32);
    }
    if (rc) return rc;
    std::memcpy(up_in.table<char>(i_ptoff), pt_off, (F + 1) * 4);
    std::memcpy(up_in.table<char>(i_scale), scale, (size_t)nlevels * 4);
    if (rule == 2) std::memcpy(up_in.table<char>(i_cam), cam, F * 7 * 4);
    WinPair* grid = up_in.table<WinPair>(i_grid);
    ProjFrame* frames = up_in.table<ProjFrame>(i_frames);
    Lists rooms;
    for (int f = 0; f < n_frames; f++) {
        const int k0 = key_off[f], q0 = pt_off[f];
        WinPair& w = grid[f];
        std::memset(&w, 0, sizeof(w));
        w.kp2 = (const OrbKeyPoint*)(d_in + i_kp) + k0;
        w.uright = (const float*)(d_in + i_ur) + k0;
        w.occupied = (const uint8_t*)(d_in + i_occ) + k0;
        w.n2 = key_off[f + 1] - k0;
        w.minX = bounds[4 * f];
        w.maxX = bounds[4 * f + 1];
        w.minY = bounds[4 * f + 2];
        w.maxY = bounds[4 * f + 3];
        w.rec = (float4*)(d_s + s_rec) + k0;
        w.cell_start = (int*)(d_s + s_cells) + (size_t)f * (64 * 48 + 1);
        ProjFrame& P = frames[f];
        std::memset(&P, 0, sizeof(P));
        P.kp = w.kp2;
        P.desc = (const uint8_t*)(d_in + i_desc) + (size_t)k0 * 32;
        P.n = w.n2;
        P.minX = w.minX;
        P.maxX = w.maxX;
        P.minY = w.minY;
        P.maxY = w.maxY;
        P.rec = w.rec;
        P.cell_start = w.cell_start;
        P.q = (ProjQuery*)(d_s + s_q) + q0;
        P.qdesc = (const uint8_t*)(d_in + i_pdesc) + (size_t)q0 * 32;
        P.nq = pt_off[f + 1] - q0;
        P.cnt = (int*)(d_s + s_cnt) + q0;
        P.off = (unsigned long long*)(d_s + s_off) + q0;
        for (int b = 0; b < 2; b++) P.out[b] = (int*)(d_s + s_out) + b * np + q0;
        for (int b = 0; b < 3; b++) P.claim[b] = (int*)(d_s + s_claim) + b * nk + k0;
        P.changed = (int*)(d_out + o_chg) + (size_t)f * ORB_PROJ_MAXIT;
        P.rule = rule;
        P.nnratio = nnratio;
        P.check_orientation = check_orientation ? 1 : 0;
        P.pt_match = (int*)(d_out + o_ptm) + q0;
        P.key_point = (int*)(d_out + o_keyp) + k0;
        P.nmatch = (int*)(d_out + o_nm) + f;
        rooms.add(P.nq, P.n);
    }
    const unsigned long long* tot = (const unsigned long long*)(h_out + o_tot);
    const int* chg = (const int*)(h_out + o_chg);
    auto place_lists = [&](size_t n) -> int {
        const int rg = reserve(ctx, &ctx->d_wcand, &ctx->wcand_cap, std::max<size_t>(n, 1) * sizeof(unsigned));
        if (rg) return rg;
        size_t start = 0;
        for (int f = 0; f < n_frames; f++) {
            frames[f].cand = (unsigned*)ctx->d_wcand;
            frames[f].room = grid[f].room =
                rooms.room(f, start, ctx->wcand_cap / sizeof(unsigned), (unsigned long long*)(d_out + o_tot));
            start += rooms.region(f);
        }
        return ORB_OK;
    };
    rc = place_lists(rooms.regions);
    if (!rc) rc = up_in.finish();
    if (rc) return rc;
    const WinPair* d_grid = (const WinPair*)(d_in + i_grid);
    ProjFrame* d_frames = (ProjFrame*)(d_in + i_frames);
    auto lists = [&]() -> int {
        HIP_TRY(orb_launch_proj_prep(d_frames, n_frames, max_nq, rule, (const float*)(d_in + i_pts),
                                     (const int*)(d_in + i_ptoff), (const float*)(d_in + i_scale), nlevels,
                                     (const float*)(d_in + i_cam), mono, th, st));
        HIP_TRY(orb_launch_proj_lists(d_grid, d_frames, n_frames, max_nq, st));
        return ORB_OK;
    };
    auto run_device = [&]() -> int {
        const int limit = std::min(ctx->round_limit, ORB_PROJ_MAXIT);
        int k = 0;
        bool settled = false;
        ctx->last_restarts = 0;
        int rl = lists();
        if (rl) return rl;
        // claim-resolution rounds until every frame has a round that changed
        // nothing, in chunks of 4, each followed by the finish of the frames
        // that have settled
        for (;;) {
            const int k1 = std::min(limit, k + 4);
            HIP_TRY(orb_launch_proj_rounds(d_frames, n_frames, max_nq, k, k1, st));
            k = k1;
            HIP_TRY(orb_launch_proj_finish(d_frames, n_frames, 0, st));
            HIP_TRY(hipMemcpyAsync(h_out, d_out, B.out, hipMemcpyDeviceToHost, st));
            HIP_TRY(hipStreamSynchronize(st));
            if (tot[F] > frames[0].room.shared_cap) {  // longer lists, from the start
                ctx->last_restarts++;
                rl = place_lists(rooms.need(tot, orb_proj_queries_per_block()));
                if (rl) return rl;
                HIP_TRY(hipMemcpyAsync(d_in + i_frames, frames, F * sizeof(ProjFrame), hipMemcpyHostToDevice, st));
                rl = lists();
                if (rl) return rl;
                k = 0;
                continue;
            }
            settled = true;
            for (int f = 0; f < n_frames && settled; f++) {
                bool s = false;
                for (int r = 1; r < k && !s; r++) s = chg[(size_t)f * ORB_PROJ_MAXIT + r] == 0;
                settled = s;
            }
            if (settled || k >= limit) break;
        }
        ctx->last_rounds = k;
        ctx->last_sequential = settled ? 0 : 1;
        if (!settled) {
            HIP_TRY(orb_launch_proj_finish(d_frames, n_frames, 1, st));
            HIP_TRY(hipMemcpyAsync(h_out, d_out, B.out, hipMemcpyDeviceToHost, st));
            HIP_TRY(hipStreamSynchronize(st));
        }
        return ORB_OK;
    };
    rc = run_device();
    if (rc) return rc;
    if (steps > 0) {        // repeats with the inputs resident in HBM (they are not modified)
        const auto t0 = std::chrono::steady_clock::now();
        for (int i = 0; i < steps; i++) {
            rc = run_device();
            if (rc) return rc;
        }
        *ms = (float)(std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count() / steps);
    }
    // (rows before the first frame's are not the call's to write)
    const size_t k0 = (size_t)key_off[0], q0 = (size_t)pt_off[0];
    if (np > q0) std::memcpy(pt_match + q0, h_out + o_ptm + q0 * 4, (np - q0) * 4);
    if (nk > k0) std::memcpy(key_point + k0, h_out + o_keyp + k0 * 4, (nk - k0) * 4);
    std::memcpy(nmatches, h_out + o_nm, F * 4);
    return ORB_OK;
}

}  // namespace

extern "C" {

int orb_context_set_round_limit(orb_context* ctx, int rounds)
{
    if (!ctx || rounds < 0 || rounds > ORB_WIN_MAXIT) return ORB_E_ARG;
    ctx->round_limit = rounds;
    return ORB_OK;
}

int orb_context_last_rounds(const orb_context* ctx, int* sequential)
{
    if (!ctx) return ORB_E_ARG;
    if (sequential) *sequential = ctx->last_sequential;
    return ctx->last_rounds;
}

int orb_context_last_restarts(const orb_context* ctx) { return ctx ? ctx->last_restarts : ORB_E_ARG; }

int orb_search_by_projection(orb_context* ctx, int n_frames, const orb_keypoint* kp, const uint8_t* desc,
                             const float* uright, const uint8_t* occupied, const int32_t* key_off,
                             const float* bounds, const float* scale_factors, int nlevels,
                             const orb_proj_point* points, const uint8_t* point_desc, const int32_t* point_off,
                             float th, float nn_ratio, int32_t* point_match, int32_t* key_point, int32_t* nmatches)
{
    return proj_search(ctx, 1, n_frames, kp, desc, uright, occupied, key_off, bounds, scale_factors, nlevels, points,
                       point_desc, point_off, nullptr, 0, th, nn_ratio, 0, point_match, key_point, nmatches, 0,
                       nullptr);
}

int orb_search_by_projection_time(orb_context* ctx, int n_frames, const orb_keypoint* kp, const uint8_t* desc,
                                  const float* uright, const uint8_t* occupied, const int32_t* key_off,
                                  const float* bounds, const float* scale_factors, int nlevels,
                                  const orb_proj_point* points, const uint8_t* point_desc, const int32_t* point_off,
                                  float th, float nn_ratio, int32_t* point_match, int32_t* key_point,
                                  int32_t* nmatches, int steps, float* ms)
{
    if (steps <= 0 || !ms) return ORB_E_ARG;
    return proj_search(ctx, 1, n_frames, kp, desc, uright, occupied, key_off, bounds, scale_factors, nlevels, points,
                       point_desc, point_off, nullptr, 0, th, nn_ratio, 0, point_match, key_point, nmatches, steps,
                       ms);
}

int orb_search_by_projection_last(orb_context* ctx, int n_frames, const orb_keypoint* kp, const uint8_t* desc,
                                  const float* uright, const uint8_t* occupied, const int32_t* key_off,
                                  const float* bounds, const float* scale_factors, int nlevels, const float* camera,
                                  int mono, const orb_last_point* points, const uint8_t* point_desc,
                                  const int32_t* point_off, float th, int check_orientation, int32_t* point_match,
                                  int32_t* key_point, int32_t* nmatches)
{
    return proj_search(ctx, 2, n_frames, kp, desc, uright, occupied, key_off, bounds, scale_factors, nlevels, points,
                       point_desc, point_off, camera, mono, th, 0.f, check_orientation, point_match, key_point,
                       nmatches, 0, nullptr);
}

int orb_search_by_projection_last_time(orb_context* ctx, int n_frames, const orb_keypoint* kp, const uint8_t* desc,
                                       const float* uright, const uint8_t* occupied, const int32_t* key_off,
                                       const float* bounds, const float* scale_factors, int nlevels,
                                       const float* camera, int mono, const orb_last_point* points,
                                       const uint8_t* point_desc, const int32_t* point_off, float th,
                                       int check_orientation, int32_t* point_match, int32_t* key_point,
                                       int32_t* nmatches, int steps, float* ms)
{
    if (steps <= 0 || !ms) return ORB_E_ARG;
    return proj_search(ctx, 2, n_frames, kp, desc, uright, occupied, key_off, bounds, scale_factors, nlevels, points,
                       point_desc, point_off, camera, mono, th, 0.f, check_orientation, point_match, key_point,
                       nmatches, steps, ms);
}

}  // extern "C"
