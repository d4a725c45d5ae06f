// orb_types.h -- job descriptors shared by the host runtime and the gfx950
// kernels of the ORB front end.
//
// One ImageJob describes one image going through the extraction pipeline
// (pyramid -> FAST cells -> quadtree distribution -> orientation + rotated
// BRIEF).  Every job carries device pointers to its own buffers, so a single
// launch of each stage can cover any set of images: the two views of a stereo
// frame, a mixed-size batch, or the frames admitted by the serving loop.
#pragma once
#include <stdint.h>

#define ORB_MAX_LEVELS 16
#define ORB_DESC_KPB 16             // keypoints per describe workgroup (16 lanes each)
#define ORB_MAX_ROOTS 16
#define ORB_LIST_CAP 1024      // quadtree list capacity per level (LDS; one node per octree thread)
#define ORB_TILE_W 64          // level kernel output tile
#define ORB_MAX_CHAINS (ORB_MAX_LEVELS - 1)
// Pyramid kernel: tile of a chain's last level (small for runs of few images,
// large for many), threads, and the most dwords, dwords a row and rows of a
// window in LDS.  Large tiles in a batch of 128 images of 1241 x 376: 96 x 48
// and 6144 dwords 151 us, 64 x 64 153, 128 x 32 155, 64 x 32 and 4096 dwords
// 175, 128 x 64 with 1024 threads 179; 2560 dwords (three chains) 161.
#define ORB_CH_VARIANTS 2
#define ORB_CH_W(v) ((v) ? 96 : 32)
#define ORB_CH_H(v) ((v) ? 48 : 16)
#define ORB_CH_T 512
#define ORB_CH_DWORDS 6144
#define ORB_CH_COLS 96
#define ORB_CH_ROWS 160
// At most this many small tiles: the small variant.  Images of 640 x 480, 8
// levels, small (one launch) against large (two): 4 images (216 small tiles)
// 15.0 us against 24.3, 8 20.8 against 25.5, 12 (648) 27.6 against 28.7, 16
// 34.5 against 31.7, 32 55.6 against 39.7.
#define ORB_CH_FEW 640
#define ORB_EDGE 19            // EDGE_THRESHOLD, ORBextractor.cc:81
#define ORB_MIN_BORDER 16      // EDGE_THRESHOLD - 3, ORBextractor.cc:1049

// Counter slots per job (int32, zeroed at the start of each run).
#define ORB_CNT_RET 16                       // [16] keypoints kept per level
#define ORB_CNT_NOUT (ORB_CNT_RET + 16)      // total keypoints
#define ORB_CNT_ERR (ORB_CNT_NOUT + 1)       // error bits
#define ORB_CNT_MATCH (ORB_CNT_ERR + 1)      // stereo matches recorded
#define ORB_CNT_SLOTS 64

// A level's candidates lie in ORB_SEGS lists, tile t appending to list t %
// ORB_SEGS, whose counters are ORB_SEG_STRIDE ints apart: a counter takes 25 ns
// an append, one after another.  level_kernel on one image of 1280 x 720 24.2
// us with a list a level, 13.2 with 16; of 640 x 480 11.4 and 9.4 (the quadtree
// reads a list per wavefront: 21.5 -> 22.7 us on two images of 1241 x 376).
#define ORB_SEGS 16
#define ORB_SEG_STRIDE 32

#define ORB_KEY_INI (1ull << 40)     // candidate of the iniThFAST pass
#define ORB_KEY_MIN (1ull << 41)     // candidate of the minThFAST pass (mostly the same pixels and more)
#define ORB_KEY_RANK ((1ull << 40) - 1)   // response and order key
#define ORB_OCT_D 6                  // quadtree passes found at once

#define ORB_ERR_KEYS 1        // candidate buffer overflow
#define ORB_ERR_LIST 2        // quadtree list overflow
#define ORB_ERR_OUT 4         // output capacity overflow

// cv::KeyPoint layout (28 bytes).
struct OrbKeyPoint {
    float x, y, size, angle, response;
    int octave, class_id;
};

struct LevelJob {
    int w, h, pitch;                 // level size and row pitch (bytes)
    int tiles_x, tiles_y;            // level kernel tiles
    unsigned txrcp;                  // ceil(2^31 / tiles_x): t / tiles_x = umulhi(2 t, txrcp)
    int nCols, nRows, wCell, hCell;  // FAST cell grid (ORBextractor.cc:1065-1071)
    unsigned wrcp, hrcp;             // ceil(2^32 / wCell), ceil(2^32 / hCell): x / cell = umulhi(x, rcp)
    int maxBorderX, maxBorderY;
    int quota;                       // mnFeaturesPerLevel[level]
    int nIni;                        // quadtree roots
    float hX;                        // root width (float, ORBextractor.cc:701)
    float scale;                     // mvScaleFactor[level]
    int root_x[ORB_MAX_ROOTS + 1];   // (int)(hX*i), i = 0..nIni
    int seg_cap;                     // capacity of each candidate list (both thresholds)
    int ncells;                      // nCols * nRows
    int list_cap;                    // kept-keypoint capacity (<= ORB_LIST_CAP)
    int rs_end;                      // level columns < rs_end: SSE2 resize rounding (else scalar)
    int bs_end;                      // level columns < bs_end: SSE2 blur-column rounding (else scalar)
    uint8_t* lvl;                    // level image
    uint8_t* blur;                   // 7x7 sigma-2 blur of the level
    uint8_t* cellflag;               // per FAST cell: has an iniThFAST survivor
    int* segs;                       // counters of the candidate lists
    unsigned long long* keys;        // candidates: response<<32 | order key | passes
    unsigned long long* keys2;       // candidates after the per-cell retry
    int* node;                       // per-candidate quadtree node (scratch)
    unsigned long long* ret;         // kept keypoints in output order
    const int2* xtab;                // levels >= 1: per column {sx | sse2 << 30, a0 | a1 << 16} of the
    const int2* ytab;                // resize from level-1; per row {sy, b0 | b1 << 16}
    const unsigned short* octx;      // quadtree place at depth ORB_OCT_D of a candidate at (x, y):
    const unsigned short* octy;      // octx[x] ^ octy[y] (x, y relative to the border)
};

// A run of pyramid levels that one launch computes, base + 1 .. base + m from
// base, a workgroup per tile of the last.  Per tile column (and row), m + 1
// entries, of base first: the first and last column a workgroup needs of the
// level (a, b), the [o0, o1) it writes, and for columns the window's dwords a
// row and ceil(2^20 / dwords).
struct ChainWin {
    int a, b, o0, o1;
    int nd;
    unsigned rcp;
    int pad[2];
};
struct ChainJob {
    int base, m;
    int tiles_x, tiles_y;
    int staged;                      // the windows fit in LDS (else m = 1, read from memory)
    const ChainWin* xr;
    const ChainWin* yr;
};

struct ImageJob {
    const uint8_t* src;              // input image (level 0), src_pitch bytes per row; the
    int src_pitch;                   // level kernel copies it into lv[0].lvl unless it is lv[0].lvl
    int nlevels, iniTh, minTh;
    int out_cap;                     // keypoint output capacity
    int* counters;                   // ORB_CNT_SLOTS ints
    OrbKeyPoint* kps;                // out_cap keypoints
    uint8_t* desc;                   // out_cap x 32 bytes
    int nchains[ORB_CH_VARIANTS];
    ChainJob ch[ORB_CH_VARIANTS][ORB_MAX_CHAINS];
    LevelJob lv[ORB_MAX_LEVELS];
};

#define ORB_MAX_JOBS 256

// Launch table for one run over a set of jobs (prefix sums in block units).
struct RunTable {
    int njobs;
    int max_levels;
    int tile_start[ORB_MAX_LEVELS][ORB_MAX_JOBS + 1];   // per level: first tile block of job j
    int desc_start[(ORB_MAX_JOBS + 1) * ORB_MAX_LEVELS];  // describe kernel: first block of (job, level)
    int tiles_per_job[ORB_MAX_LEVELS];  // > 0: every job has this many tiles at the level,
    unsigned tiles_rcp[ORB_MAX_LEVELS]; // and block / tiles = umulhi(2 block, ceil(2^31 / tiles))
    int tile_h[ORB_MAX_LEVELS];         // level kernel tile height at the level (32 or 16)
    int all_start[2][ORB_MAX_LEVELS + 1];   // one launch for the levels of tile height 32 / 16: first block of each
    int chain_variant;                  // of the jobs' chains
    int nchains;                        // pyramid launches
    int chain_start[ORB_MAX_CHAINS][ORB_MAX_JOBS + 1];   // per pyramid launch: first block of job j
    int chain_per_job[ORB_MAX_CHAINS];  // > 0: every job has this many blocks
    int chain_zeroes;                   // the first pyramid launch has a block for every job, and clears its counters
    int desc_per_job;                   // > 0: every job has this many describe blocks
};

// Arguments of one stereo match (Frame::ComputeStereoMatches).
struct StereoArgs {
    const ImageJob* left;
    const ImageJob* right;
    const OrbKeyPoint* kl;
    const uint8_t* dl;
    const int* nl;
    const OrbKeyPoint* kr;
    const uint8_t* dr;
    const int* nr;
    int cap_l;
    int nrows;
    float bf, mb;
    float scale[ORB_MAX_LEVELS], inv_scale[ORB_MAX_LEVELS];
    float* uRight;
    float* depth;
    int* match_sad;         // per left keypoint: SAD of its match, or -1
    int4* srec;             // scratch: right keypoints grouped by row bucket as
                            // {minr, maxr, index << 4 | octave, x bits} ...
    uint8_t* sdesc;         // ... and their descriptors in the same order
    int2* rows;             // per (octave o, level-0 row): [first, end) of the entries
                            // of octave o whose row band can hold the row (nlev x nrows)
    int cap_r;
    int nlev;               // pyramid levels of both extractors
};

// Arguments of one brute-force match of a query set against a train set
// (serving: this frame's descriptors against the stream's previous ones).
struct MatchArgs {
    const uint8_t* q;
    const int* nq;
    const uint8_t* t;
    const int* nt;
    int th_low;
    float ratio;
    int* idx;
    int* dist;
    int cap_q;
    int wave_base;          // first wavefront of this pair in a multi-pair launch
    uint8_t* save_desc;     // after matching: q copied here ...
    int* save_n;            // ... and *nq here (the stream's resident state)
    int save_cap;
};

// One region of a batch's staged host transfers, copied in 4-byte words:
// `words` of them, or min(words, *count * unit_words) when count is set (a
// slot's keypoint count, read on the device).  Source and destination are
// 4-byte aligned; a region that is a whole number of 16-byte words at
// 16-byte aligned addresses is copied 16 bytes at a time.  Either side may
// be pinned host memory, which the device reads and writes over PCIe.
struct CopyOp {
    const unsigned* src;
    unsigned* dst;
    const int* count;
    int words;
    int unit_words;
};

// A copy list short enough to be a kernel argument.
#define ORB_COPY_LIST 8
#define ORB_COPY_BLOCKS 16            // workgroups an operation of a single call's list
struct CopyList {
    CopyOp op[ORB_COPY_LIST];
    int n;
};

// A DBoW2 vocabulary tree on the device, nodes renumbered breadth-first so
// that every node's children are contiguous (in their file order).
struct VocDev {
    const int2* meta;       // per node: first child, number of children
    const uint4* desc;      // per node: 32-byte descriptor as two uint4
    const int* orig_id;     // per node: id in the file (node 0 = root)
    const int* word_id;     // per node: word id (0 for non-words)
    const double* weight;   // per node: weight from the file
    int n_nodes;
    int L;                  // depth levels from the header (nid level = L - levelsup)
    int max_depth;          // deepest node, bounds every descent
    int scoring, weighting;
};

// One image of a BoW batch: its rows [off, off + n) of the descriptor and
// per-descriptor arrays; outputs at the same offsets.
struct BowJob {
    int off, n;
};

// Where a frame's (or pair's) candidate lists go in the call's buffer: a region
// of its own, and past that the end of the buffer, which the frames share.
// Counters are of entries asked for, on the device.
struct ListRoom {
    unsigned long long* asked;         // of this frame
    unsigned long long* asked_shared;  // of the shared part (beyond shared_cap: lists are missing)
    unsigned long long start, cap;     // the region
    unsigned long long shared_start, shared_cap;
};

// One frame pair of ORBmatcher::SearchForInitialization: F1 / F2 keypoints
// (mvKeysUn) and descriptors, the grid bounds (mnMinX .. mnMaxY), the search
// positions (vbPrevMatched), parameters, scratch and
// outputs.
struct WinPair {
    const OrbKeyPoint* kp1;
    const uint8_t* d1;
    const OrbKeyPoint* kp2;
    const uint8_t* d2;
    int n1, n2;
    float minX, maxX, minY, maxY;
    const float2* prev;
    int window;
    float nnratio;
    int check_orientation;
    // the grid's keypoints sorted by (cell, index): x, y, mvuRight,
    // index | octave << 12; only keypoints a query can take (below)
    float4* rec;
    int* cell_start;        // 64*48 + 1
    const float* uright;    // SearchByProjection's frames: mvuRight and occupancy
    const uint8_t* occupied;   // (occupied keypoints are left out); null: octave 0 only
    int* cnt;               // n1: candidates per query
    unsigned long long* off;     // n1: where each query's list starts in cand
    int2* cand;             // (i2, distance) lists of the whole call
    ListRoom room;
    int* m12;               // n1: vnMatches12
    float2* prev_out;       // n1: vbPrevMatched afterwards
    int* nmatch;            // nmatches
    // SearchForInitialization's in-order pass as parallel rounds (unused by
    // the grid kernels of SearchByProjection, which leave them null)
    int* out[2];            // n1 per round parity: accepted target << 9 | distance, or -1
    unsigned* claim[3];     // n2 * ORB_WIN_SLOTS per round mod 3: query << 9 | distance
    int* ccnt[3];           // n2 per round mod 3: claims written (beyond ORB_WIN_SLOTS: overflow)
    int* changed;           // [ORB_WIN_MAXIT]: bit 0 an outcome changed, bit 1 claims overflowed,
                            // bit 2 the round has not run
};
#define ORB_WIN_MAXIT 48
#define ORB_WIN_SLOTS 8

// ORBmatcher::SearchByProjection: one query (a map point to place in the
// frame) after the per-point arithmetic of either overload.
struct ProjQuery {
    float x, y, r;          // window centre and radius (GetFeaturesInArea)
    float su;               // right-image u compared with mvuRight (radius r)
    int minL, maxL;         // GetFeaturesInArea level arguments
    int flags;              // ORB_PQ_VALID | ORB_PQ_OBS
    float angle;            // last-frame keypoint angle (rotation check)
};
#define ORB_PQ_VALID 1
#define ORB_PQ_OBS 4
#define ORB_PROJ_MAXIT 48   // claim-resolution rounds before the sequential pass

// One frame of a SearchByProjection call: its keypoints (mvKeysUn),
// descriptors, mvuRight, occupancy and grid, the queries, their candidate
// lists, and the claim-resolution state.
struct ProjFrame {
    const OrbKeyPoint* kp;
    const uint8_t* desc;
    int n;
    float minX, maxX, minY, maxY;
    const float4* rec;          // grid, as WinPair's
    const int* cell_start;
    ProjQuery* q;
    const uint8_t* qdesc;
    int nq;
    int* cnt;                   // candidates per query
    unsigned long long* off;    // where each query's list starts in cand
    unsigned* cand;             // i2 | distance << 12 | octave << 21, GetFeaturesInArea order
    ListRoom room;
    int* out[2];                // outcome per query by round parity: keypoint or -1
    int* claim[3];              // per keypoint: first claiming query (with observations), by round mod 3
    int* changed;               // [ORB_PROJ_MAXIT]: bit 0 round k changed some outcome, bit 2 not run
    int rule;                   // 1: local map (best + second, level ratio); 2: last frame (best, rotation)
    float nnratio;
    int check_orientation;
    int* pt_match;              // outputs
    int* key_point;
    int* nmatch;
};
