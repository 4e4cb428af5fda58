// upbp_internal.hpp -- host-side objects behind the opaque handles of include/upbp.h.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <string>
#include <vector>

#include "../../include/upbp.h"
#include "upbp_device.hpp"
#include "beamgrid.hpp"

namespace upbp {

// Error carried from a failing HIP call up to the C ABI.
struct Error {
    upbp_status status;
    std::string message;
};

#define UPBP_HIP(call)                                                                       \
    do {                                                                                     \
        hipError_t e_ = (call);                                                              \
        if (e_ != hipSuccess) {                                                              \
            throw ::upbp::Error{e_ == hipErrorOutOfMemory ? UPBP_ENOMEM : UPBP_EDEVICE,      \
                                std::string(#call) + ": " + hipGetErrorString(e_)};         \
        }                                                                                    \
    } while (0)

#define UPBP_REQUIRE(cond, status, msg)                  \
    do {                                                 \
        if (!(cond)) throw ::upbp::Error{(status), (msg)}; \
    } while (0)

// Owning device buffer (hipMalloc / hipFree), grows on demand.
struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf() { release(); }
    void release() {
        if (p) (void)hipFree(p);
        p = nullptr;
        bytes = 0;
    }
    void ensure(size_t n) {
        if (n <= bytes) return;
        release();
        size_t want = n < 256 ? 256 : n;
        UPBP_HIP(hipMalloc(&p, want));
        bytes = want;
    }
    template <class T>
    T* as() const { return static_cast<T*>(p); }
};

// Build temporaries: grow-only device buffers that a context keeps and lends out for one scope
// at a time, last borrowed first returned (every call on a context runs on its one stream, and
// a context is used by one host thread at a time). A renderer that rebuilds its structures every
// iteration then allocates and frees no temporary device memory once the sizes are reached; the
// buffers are freed with the context.
struct TmpPool {
    static constexpr int kSlots = 48;
    DevBuf slot[kSlots];
    int top = 0;
};

class TmpBuf {
  public:
    explicit TmpBuf(TmpPool& pool) : pool_(pool), b_(take(pool)), p(b_.p) {}
    ~TmpBuf() { --pool_.top; }
    TmpBuf(const TmpBuf&) = delete;
    TmpBuf& operator=(const TmpBuf&) = delete;
    void ensure(size_t n) { b_.ensure(n); }
    template <class T>
    T* as() const { return b_.as<T>(); }
    operator DevBuf&() { return b_; }

  private:
    static DevBuf& take(TmpPool& pool) {
        UPBP_REQUIRE(pool.top < TmpPool::kSlots, UPBP_EDEVICE, "build temporaries exhausted");
        return pool.slot[pool.top++];
    }
    TmpPool& pool_;
    DevBuf& b_;

  public:
    void*& p;  // the lent buffer's pointer (follows ensure)
};

// Counters written by the traversal kernels (device, uint64 each).
enum StatSlot : int {
    kStatPhotonHits = 0,
    kStatBeamHits = 1,
    kStatPhotonCands = 2,
    kStatBeamCands = 3,
    kStatNodes = 4,
    kStatError = 5,     // bit mask of input errors found by kernels
    kStatOverflow = 6,  // traversal stack overflow count
    kStatSlots = 8
};
// The counters are kept in kStatRows rows of kStatSlots (one 64-byte line each) that the waves
// spread over, added up by the host (sum_stats): with one row every wave of a launch queued for
// the same few words. 131072 waves that had almost nothing else to do took 1.9 ms.
constexpr int kStatRows = 64;
constexpr int kStatWords = kStatRows * kStatSlots;

// What the kernels of a tile plan count (traverse.hip), cleared with the counters.
struct PlanWords {
    unsigned long long total[64][2];  // cost and number of the tiles with an estimate, spread over rows
    uint32_t n_tasks, n_rows;
    uint32_t hist[64], cursor[64];
};
constexpr int kStatAll = kStatWords + 2 * (int)(sizeof(PlanWords) / 8);  // with both estimators' plan words

inline void sum_stats(const uint64_t* rows, uint64_t* st) {
    for (int k = 0; k < kStatSlots; ++k) st[k] = 0;
    for (int r = 0; r < kStatRows; ++r)
        for (int k = 0; k < kStatSlots; ++k) {
            const uint64_t v = rows[r * kStatSlots + k];
            st[k] = k == kStatError ? (st[k] | v) : st[k] + v;
        }
}
constexpr uint32_t kErrBadOffsets = 1u, kErrBadMedium = 2u, kErrBadSegment = 4u, kErrNonFinite = 8u;

struct Tuning {
    int waves_per_block = 4;
    int blocks_per_cu = 0;
    int photon_waves_per_block = 0;  // 0: waves_per_block
    int frustum_leaf = 64;           // largest subtree a frustum wave tests as one leaf
};

struct Ctx {
    // References: the caller's (dropped by upbp_ctx_destroy) plus one per photon
    // structure, beam structure and batch plan built on this context.
    std::atomic<int> refs{1};
    int device = 0;
    hipStream_t own_stream = nullptr;
    hipStream_t stream = nullptr;
    bool sync = true;
    std::string last_error;
    int n_media = 0;
    std::vector<MediumDev> media_host;
    DevBuf media;
    // sign of every input coefficient (+1 / -1) as [M][6] floats (absorption RGB, scattering RGB):
    // the media use |sigma| (Media.hxx:136-140), so gradients with respect to the caller's
    // values carry these factors
    DevBuf media_sign;
    std::vector<float> media_sign_host;
    // bumped by every upbp_set_media: a batched plan whose captured graph froze an older table
    // re-validates its instances and captures again
    uint64_t media_gen = 0;
    DevBuf stats;       // kStatAll x uint64
    DevBuf sort_tmp;    // hipcub temporary storage
    TmpPool tmp;        // build temporaries
    DevBuf qkeys, qkeys2, qperm, qperm2;
    DevBuf light_tails;  // float4 per light vertex of the current UPBP call
    DevBuf beam_recs;    // 64-byte MIS record per photon beam of the current UPBP call
    DevBuf photon_recs;  // 64-byte MIS record per light vertex of the current UPBP call
    DevBuf vm_rec;       // merge records (4 float4 per grid slot) of the current PP3D / SURF call
    DevBuf lt_slots[8];  // light tracing: per-path vertex, position and beam slots, counts, offsets, lights
    DevBuf plan[2];  // a split evaluation's plan and rows, per estimator
    DevBuf staging[8];  // host-input staging copies
    hipEvent_t ev[6] = {};
    // second stream: the photon and beam kernels of one eval call run concurrently
    // (fork from `stream`, join back), so one kernel's tail overlaps the other's work
    hipStream_t side = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
    // An evaluation that returned before its work ended, and the end of that work: the next one, which may
    // be on another stream (upbp_ctx_set_stream), waits for it, as both work in the buffers above.
    bool in_use = false;
    hipEvent_t used = nullptr;
    // resident blocks per CU of the two persistent batched kernels at batched_key waves per block
    int batched_key = 0;
    int batched_per_cu[2] = {0, 0};
    int num_cus = 256;
    Tuning tuning;
    // this device's copy of the allocation-free entry point's fixed region (null: lookup failed)
    void* scratch = nullptr;
    std::string scratch_error;
};

// A built LBVH: node array plus the item order it implies.
struct Lbvh {
    DevBuf nodes;
    int64_t n_nodes = 0;
    int64_t n_items = 0;
    float lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};  // bounds of all item boxes
};

struct Bre {
    Ctx* ctx = nullptr;
    int64_t n_in = 0;  // photons given to build
    int64_t n = 0;     // kept photons
    Lbvh bvh;
    DevBuf pos_r2;  // float4 [n]
    DevBuf power;   // float4 [n]
    DevBuf inc;     // float4 [n]
    DevBuf orig;    // uint32 [n] original input index
    DevBuf radius_in;  // float [n_in] radius the build gave each input photon (0 if filtered out)
};

struct Beams {
    Ctx* ctx = nullptr;
    int64_t n = 0;        // beams
    int64_t pieces = 0;   // beam pieces in the LBVH
    Lbvh bvh;
    DevBuf piece;         // PieceDev [pieces]
    DevBuf piece_flux;    // float4 [pieces] throughput (rgb, 0)
    DevBuf piece_beam;    // uint32 [pieces] original beam index
    DevBuf end_bits;      // a bit per piece, in uint64 words and one more: a beam's first or last
    DevBuf r_start, r_end;  // float [n] start / end radius the build gave each beam
    // per-cell beam reduction (max_beams_in_cell > 0): the reference grid's cell lists
    RedDev red;            // device view; red.max == 0 without reduction
    int64_t red_cells = 0;
    DevBuf red_off, red_ids, red_rank;
    // the grid's box top and cell size (with red_cells > 0), and the resolution the build was
    // given (0 = 256): what a walk of the grid needs besides RedDev
    float grid_hi[3] = {0.f, 0.f, 0.f}, grid_cell[3] = {0.f, 0.f, 0.f};
    int32_t grid_resolution = 0;
};

// How the items of a batch's tiles are split over waves (split_of): uniformly over 2^log_parts, or by a
// plan that gives a tile up to 2^log_most parts.
struct Split {
    int64_t tiles = 0, waves = 0;
    uint32_t log_parts = 0, log_most = 0;
    bool planned = false;
    int64_t rows = 0;  // sums of parts kept for k_sum_rows, 64 x 3 floats each
    // whether the launch has the tuned number of waves per block (launch_waves chooses for the others)
    bool whole() const { return log_parts == 0 && !planned; }
};

// Device memory of a split: the rows, and of a plan the tiles' costs, their part counts and first rows,
// and the tasks.
struct TilePlan {
    uint32_t* cost = nullptr;
    uint2 *info = nullptr, *tasks = nullptr;
    PlanWords* words = nullptr;
    float* rows = nullptr;
    static size_t bytes(const Split& s) {
        return (size_t)s.rows * 768 + (s.planned ? (size_t)s.tiles * 20 + (size_t)s.waves * 8 : 0);
    }
    // lays the plan of s out in bytes(s) of memory at p (256-byte aligned)
    static TilePlan at(const Split& s, char* p) {
        TilePlan t;
        t.rows = reinterpret_cast<float*>(p);
        if (s.planned) {
            t.tasks = reinterpret_cast<uint2*>(p + (size_t)s.rows * 768);
            t.info = t.tasks + (s.tiles + s.waves);
            t.cost = reinterpret_cast<uint32_t*>(t.info + s.tiles);
        }
        return t;
    }
};

// Device memory one evaluation works in besides its inputs and outputs: the kernels' counters,
// the Morton keys and permutations of the query sort and the sort's temporary storage. The
// context's own growable buffers by default; the allocation-free entry point passes a fixed
// region instead.
struct Workspace {
    unsigned long long* stats = nullptr;  // kStatAll words: kStatWords counters, two PlanWords
    uint32_t *keys = nullptr, *keys2 = nullptr, *perm = nullptr, *perm2 = nullptr;  // [max_sorted] each
    int64_t max_sorted = 0;
    void* sort_tmp = nullptr;
    size_t sort_tmp_bytes = 0;
    TilePlan plan[2];  // per estimator
};

// Device-resident view of a query batch.
struct QueryView {
    int64_t count = 0;
    const float* origin = nullptr;
    const float* direction = nullptr;
    const int64_t* offsets = nullptr;
    const upbp_volume_segment* segments = nullptr;
    uint32_t beam_type = UPBP_LONG_BEAM;
    uint32_t lite = 0;
    const uint32_t* perm = nullptr;  // lane slot -> query index, or null (identity)
    // per estimator
    Split split[2];
    TilePlan plan[2];
};

// A tile of 64 queries is one wave, and the GPU holds 8192 of them: a batch of fewer tiles leaves it
// partly idle, and one of a few times more waits for the waves that meet most of the items. So a
// tile's items are split over as many waves as bring the launch to kSplitWaves, at most kSplitMost, each
// for at least kSplitItems items. Structures of fewer than kSplitFrom items stay whole: little is left to
// split there, and their sums stay the same bits as a batched plan's, which leaves them whole too. Every part
// walks the top of the tree again, so photons, which are tested in less time than beams, and the UPBP
// kernels, of which the GPU holds half as many waves, stop at kSplitWavesLight. Measured unsplit / at
// 4096 / 8192 / 16384 / 32768 waves for every estimator:
//   64x36 rays x 20k photons + 2k beams       820 /  206 /  220 /  212 /  213 us
//   256x256 rays x 100k photons               282 /  216 /  231 /  250 /  326 us
//   512x512 rays, forward and adjoint        9.73 / 9.80 / 9.99 / 9.00 / 10.1 ms
//   640x360 rays x 40k traced beams          21.6 / 21.9 / 14.8 /  8.6 /  6.6 ms
//   60k rays x 300k beams                    13.0 /  6.9 /  4.7 /  4.4 /  3.8 ms
//   200k rays without a common origin        17.2 / 16.9 / 16.8 / 14.5 / 14.6 ms
//   300x168 rays, UPBP                        699 /  445 /  504 /  637 /  892 us
// Above that many tiles nothing is split without a plan: 1920x1080 rays took 12.4 ms either way at 2
// parts, 13.7 at 4.
constexpr int64_t kSplitWaves = 16384, kSplitWavesLight = 4096;
constexpr int64_t kSplitItems = 256, kSplitFrom = 16384;
constexpr uint32_t kSplitMost = 64;

// From kPlanTiles to kPlanMostTiles tiles (2^21 queries) a beam launch plans: a tile gets as many of
// kPlanWaves waves, at most kPlanMost, as its share of the estimated cost, and the dearest parts start
// first. Estimating takes 50 to 610 us alone (6250 to 32400 tiles) and runs next to the photon kernel in
// calls with both; fewer tiles do not earn it back (256x256 rays x 100k photons
// 220 -> 270 us with 1024 tiles; photons and the UPBP kernels gain nothing and don't plan). Above
// kPlanFewTiles tiles kSplitWaves, so that average tiles stay whole. Measured uniform / planned with
// 16384 / 24576 / 32768 waves:
//   640x360 rays x 40k traced beams          7.99 / 3.92 / 3.83 / 3.88 ms
//   512x512 rays, forward and adjoint        9.00 / 9.14 / 8.60 / 8.92 ms
//   60k rays x 300k beams                    4.37 / 4.13 / 3.49 / 3.41 ms
//   400x241 rays x 200k photons + 40k beams  1.10 / 1.06 / 0.96 / 1.00 ms
//   1M rays x 2M beams                       45.8 / 38.8 / 41.6 / 41.7 ms
//   1920x1080 rays x 125k traced beams       88.0 / 23.0 ms
//   1600x900 rays x 25k traced beams         20.8 / 6.07 ms
//   1920x1080 rays x 1M photons, 200k beams  9.02 / 8.57 ms (8.04 / 8.71 at waves_per_block 1)
//   1500x1001 rays x 500k photons, 20k beams 2.02 / 2.09 ms
constexpr uint32_t kPlanMost = 256;
constexpr int64_t kPlanTiles = 512, kPlanMostTiles = 32768, kPlanFewTiles = 8192, kPlanWaves = 24576;
// Batched plans of this many tiles are planned too, both estimators, with kPlanWaves waves. Tiles of small
// instances stay whole there; the order alone shortens the tail. Instances whose tiles cost alike gain
// nothing and pay for the estimates (0.2 to 0.4 ms). Measured in queue order / planned:
//   16 instances, 4.6M rays                  6.86 / 3.81 ms
//   18 instances x 26k rays                  5.98 / 1.45 ms
//   5 instances x 22k rays                   1.92 / 0.74 ms
//   15 instances x 358k rays                 3.23 / 2.93 ms
//   8 even instances x 100k camera rays      0.63 / 0.85 ms
//   8 even instances x 100k scattered rays   2.84 / 3.23 ms
constexpr int64_t kPlanBatchTiles = 1024, kPlanBatchMost = 1 << 20;

// ---- lbvh.hip -------------------------------------------------------------
// Builds an LBVH over n item boxes (lo/hi as float4 .xyz). On return
// out_order[k] is the input index of the k-th item in leaf order.
void build_lbvh(Ctx& ctx, int64_t n, const float4* box_lo, const float4* box_hi, int leaf_size,
                Lbvh& out, DevBuf& out_order);
void sort_pairs_u64(Ctx& ctx, uint64_t* keys_in, uint64_t* keys_out, uint32_t* vals_in,
                    uint32_t* vals_out, int64_t n, int end_bit);
void sort_pairs_u32(Ctx& ctx, uint32_t* keys_in, uint32_t* keys_out, uint32_t* vals_in,
                    uint32_t* vals_out, int64_t n, int end_bit);
void exclusive_scan_u32(Ctx& ctx, const uint32_t* in, uint32_t* out, int64_t n);
// The same sort in caller-provided temporary storage (UPBP_EDEVICE if tmp_bytes is too small);
// sort_pairs_u32_temp_bytes is what it needs for n keys (no device work, no allocation).
size_t sort_pairs_u32_temp_bytes(int64_t n, int end_bit);
void sort_pairs_u32_in(Ctx& ctx, void* tmp, size_t tmp_bytes, uint32_t* keys_in, uint32_t* keys_out,
                       uint32_t* vals_in, uint32_t* vals_out, int64_t n, int end_bit);

// ---- knn.hip --------------------------------------------------------------
// Point LBVH answering "squared distance to the k-th nearest point" queries.
// Its memory is the context's build temporaries, for the object's lifetime.
struct KnnIndex {
    int64_t n = 0;
    Lbvh bvh;
    TmpBuf points;  // float4 [n] in leaf order
    explicit KnnIndex(Ctx& ctx);
    ~KnnIndex();
    // points: device xyz [*][3]; keep: optional device index list of the points to use
    void build(Ctx& ctx, int64_t n_points, const float* pts, const uint32_t* keep);
    // out[i] (device) = k-th smallest squared distance from q[i] (device xyz) to the points;
    // with n <= k the largest of the n.
    void kth_d2(Ctx& ctx, int64_t nq, const float* q, int k, float* out);

  private:
    TmpBuf nodes_;  // lends bvh.nodes its memory
};
// KNN_RADIUS of EmbreeBre::build: out_radius[i] (device, [n_in]) = radius * 2 sqrt(d2_k)
// for the kept photons (keep: kept -> input index, or null for all).
void photon_knn_radius(Ctx& ctx, int64_t n_kept, const float* pos, const uint32_t* keep, float radius, int knn,
                       DevBuf& out_radius, int64_t n_in);
// KNN_RADIUS of PhotonBeamsEvaluator::build: start / end radius per beam (device).
void beam_knn_radius(Ctx& ctx, int64_t n, const float* origin, const float* dir, const float* length, float radius,
                     int knn, DevBuf& r0, DevBuf& r1);

// ---- build.hip ------------------------------------------------------------
void bre_build(Ctx& ctx, const upbp_photon_input& in, const upbp_build_params& params, Bre& out);
void bre_set_power(Bre& bre, const float* power_dev);
void beams_build(Ctx& ctx, const upbp_beam_input& in, const upbp_build_params& params, Beams& out);

// ---- beamgrid.hip ---------------------------------------------------------
// Registers the beams (device arrays, input order) in the reference's uniform grid and
// keeps each cell's beam list and reduction ranks in out.red*; a no-op without reduction.
// With `always`, the grid is built even without reduction (red.max stays 0).
void beam_reduction_build(Ctx& ctx, int64_t n, const float* origin, const float* dir, const float* length,
                          const float* r_start, const float* r_end, const upbp_build_params& params, Beams& out,
                          bool always = false);
// Per-query GridStats of the reference grid's walk (beams tested, cells crossed, overfull
// cells crossed) into out [q.count][3] on the device (query order as given). Beams built
// without reduction get a grid of their build's resolution for the call.
void beam_grid_stats(Ctx& ctx, const Beams& b, const QueryView& q, uint32_t* out);
// Selection pdf of the cell holding pos (1 without reduction).
float beam_selection_pdf(const Beams& b, const float pos[3]);
// The same for n positions (xyz [n][3]) into out [n], both in `mem`.
void beam_selection_pdfs(const Beams& b, const float* pos, int64_t n, float* out, upbp_memory mem);

// ---- traverse.hip ---------------------------------------------------------
// EmbreeBre::evalBreBruteForce per query (device arrays; out [count][3]).
void bre_eval_brute_force(Ctx& ctx, const Bre& b, const float* origin, const float* direction, const float* min_t,
                          const float* max_t, const int32_t* medium, int64_t count, float* out);

enum class Mode : int { Forward = 0, Signature = 1, Adjoint = 2, Upbp = 3 };

struct PhotonArgs {
    const NodeDev* nodes;
    const float4* pos_r2;
    const float4* power;
    const float4* inc;
    const uint32_t* orig;
    int64_t n;
    // UPBP mode: the reduction grid of the photon-beam evaluator of the same call (sel.max == 0:
    // none), whose cell pdf at a PB2D hit is the camera vertex's BB1D beam selection pdf
    RedDev sel;
};
struct BeamArgs {
    const NodeDev* nodes;
    const PieceDev* pieces;
    const float4* piece_flux;
    const uint32_t* piece_beam;
    const uint64_t* end_bits;
    int64_t pieces_n;
    RedDev red;
};
// Rows of medium gradients that the adjoint's waves spread their atomics over (each wave adds 6 values
// per medium: on one row they queue for the same words), a power of two: up to kGradRows, and for a table
// of more than 1024 media as few as keep them all within 1.5 MB (64 rows of a million would be 1.5 GB).
constexpr int kGradRows = 64;
constexpr int64_t kGradRowMedia = 65536;
inline int grad_rows(int64_t n_media) {
    int rows = kGradRows;
    while (rows > 1 && rows * n_media > kGradRowMedia) rows /= 2;
    return rows;
}
struct AdjointOut {
    const float* grad_out;  // [Q][3]
    float* grad_media;      // [grad_rows(M)][M][6]: dsigma_s direct (0..2), dsigma_t (3..5)
    float* grad_items;      // photon [n_in][3] or beam [n][3]
};

// UPBP mode inputs on the device (upbp_mis_inputs after staging).
struct MisDev {
    const upbp_query_mis* queries;
    const upbp_mis_data* camera;
    int64_t camera_count;
    const upbp_light_vertex* lv;
    int64_t lv_count;
    const int32_t* path_ends;
    int64_t path_count;
    const upbp_beam_mis* beams;
    upbp_mis_params params;
    const float4* tails = nullptr;      // per light vertex, launch_light_tails
    const void* beam_recs = nullptr;    // per photon beam, launch_beam_records
    const void* photon_recs = nullptr;  // per light vertex, launch_photon_records
};

// stats: the kStatWords counters the kernels add to (null: the context's own)
void launch_photons(Ctx& ctx, Mode mode, const PhotonArgs& ph, const QueryView& q, float* out,
                    uint32_t* sig, const AdjointOut* adj, const MisDev* mis = nullptr,
                    unsigned long long* stats = nullptr);
void launch_beams(Ctx& ctx, Mode mode, const BeamArgs& bm, const QueryView& q, float* out,
                  uint32_t* sig, const AdjointOut* adj, const MisDev* mis = nullptr,
                  unsigned long long* stats = nullptr);
constexpr int kQueryKeyBits = 31;  // sort keys of launch_query_keys
void launch_query_keys(Ctx& ctx, const QueryView& q, const float* lo, const float* hi, bool by_direction,
                       uint32_t* keys, uint32_t* idx);
// Folds each light vertex's light walk below it into a float4 (the O(1) light walk of the
// UPBP weights) into ctx.light_tails and points mis.tails at it; nothing for no vertices.
void launch_light_tails(Ctx& ctx, MisDev& mis);
// Gathers each photon beam's MIS inputs (its record, origin light vertex and that vertex's tail)
// into ctx.beam_recs and points mis.beam_recs at it; after launch_light_tails.
void launch_beam_records(Ctx& ctx, MisDev& mis, int64_t n_beams);
// The same per light vertex for the PB2D hits into ctx.photon_recs (mis.photon_recs).
void launch_photon_records(Ctx& ctx, MisDev& mis);
// How an evaluation of count queries against items items is split: into how many parts a tile's items go, or
// whether a plan decides that tile by tile, and how many rows of partial sums that takes.
Split split_of(int64_t count, int64_t items, int estimator, Mode mode);
// Adds up a split evaluation's parts into the outputs (null: not evaluated), in query order.
void launch_sum_rows(Ctx& ctx, const QueryView& q, float* ph, float* bm);
void launch_sum_rows_sig(Ctx& ctx, const QueryView& q, uint32_t* ph, uint32_t* bm);
void launch_clear_u64(Ctx& ctx, uint64_t* p, int64_t n);
void launch_clear_f32(Ctx& ctx, float* p, int64_t n);
// gs += sign_s * (direct + d/d sigma_t), ga += sign_a * d/d sigma_t per medium and channel, summed
// over the grad_rows rows of gm (sign: [M][6] of ctx.media_sign).
void launch_combine_media_grads(Ctx& ctx, const float* gm, const float* sign, int n_media, float* gs, float* ga);

// ---- hashgrid.hip: vertex-merging hashed grid (PP3D, SURF) --------------------
struct HashGrid {
    Ctx* ctx = nullptr;
    uint32_t type = 0;  // UPBP_PP3D (in-medium vertices) or UPBP_SURF (surface vertices)
    int64_t n_src = 0;  // light vertices given to the build
    int64_t n = 0;      // vertices in the grid
    int64_t cells = 0;  // hash buckets
    float radius = 0.f, r2 = 0.f, inv_cell = 0.f;
    float lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
    DevBuf slots;  // float4 [n]: position, light-vertex index (bits); bucket order
    DevBuf slot_of;  // uint32 [n_src]: the slot of each light vertex, all ones outside the grid
    DevBuf ends;   // uint32 [cells]: one past each bucket's last slot
};
// flags[i * stride] holds the UPBP_LV_* word of light vertex i (device pointers).
void hash_grid_build(Ctx& ctx, const float* pos, const uint32_t* flags, int64_t stride, int64_t n, float radius,
                     int64_t cells, uint32_t type, HashGrid& out);
void pp3d_eval(Ctx& ctx, const HashGrid& grid, const upbp_pp3d_query* q, int64_t count, const MisDev& mis,
               uint32_t flags, float* out, uint32_t* sig);
void surf_eval(Ctx& ctx, const HashGrid& grid, const upbp_surf_query* q, int64_t count, const MisDev& mis,
               uint32_t flags, float* out, uint32_t* sig);

// ---- batched persistent kernels --------------------------------------------
struct InstanceDev {
    const NodeDev* ph_nodes;
    const float4* ph_pos_r2;
    const float4* ph_power;
    const float4* ph_inc;
    const NodeDev* bm_nodes;
    const PieceDev* bm_pieces;
    const float4* bm_flux;
    const float* origin;
    const float* direction;
    const int64_t* offsets;
    const upbp_volume_segment* segments;
    const uint32_t* perm;
    float* out_photons;
    float* out_beams;
    int64_t count;
    int64_t tile_begin;  // first global tile of this instance
    int32_t media_base;
    uint32_t beam_type;
    uint32_t lite;
    int32_t has_photons;
    int32_t has_beams;
    uint32_t ph_root;  // root of this instance's photon tree in the plan's merged node array
    uint32_t bm_root;  // root of its beam tree in the merged beam node array
    uint32_t ph_log_most, bm_log_most;  // log2 of the most parts its tiles may be split into
    uint32_t ph_group, bm_group;        // subtrees of at most this many items are estimated as one
    int32_t pad;
};

// A batched plan's copy of every instance's structures, one array each, so that the
// persistent kernel reads them through kernel-argument pointers (scalar loads).
// Child references are rebased: inner refs by the instance's node offset, leaf refs
// by its item offset.
struct MergedDev {
    const NodeDev* ph_nodes;
    const float4* ph_pos_r2;
    const float4* ph_power;
    const float4* ph_inc;
    const NodeDev* bm_nodes;
    const PieceDev* bm_pieces;
    const float4* bm_flux;
};
void launch_rebase_nodes(Ctx& ctx, NodeDev* nodes, int64_t n, uint32_t node_off, uint32_t item_off);

// Queries (outside any graph capture) how many blocks of each persistent kernel fit on a CU.
void prepare_batched(Ctx& ctx, int waves_per_block, bool planned);
// How a batched plan's tiles are split, with the memory of each estimator's tile plan. A tile of an
// instance with fewer than kSplitFrom items stays whole (batched_log_most).
struct BatchSplit {
    bool planned = false;
    TilePlan plan[2];
};
uint32_t batched_log_most(int64_t items);
void launch_batched_plan(Ctx& ctx, const InstanceDev* inst, int n_inst, int64_t total_tiles, const BatchSplit& split,
                         const MergedDev& merged, int which);
void launch_batched(Ctx& ctx, const InstanceDev* inst, int n_inst, int64_t total_tiles, uint32_t* counters,
                    const BatchSplit& split, const MergedDev& merged, int which, int grid_blocks, int waves_per_block);
void launch_fill_u32(Ctx& ctx, uint32_t* p, uint32_t v, int64_t n);

// ---- lighttrace.hip: light sub-path tracing in media ---------------------------
// Fills out (device memory) and its counts; UPBP_EINVAL when a capacity is exceeded.
void trace_light_paths(Ctx& ctx, const upbp_region* regions, int32_t n_regions, const upbp_point_light* lights,
                       int32_t n_lights, const upbp_light_trace_params& P, int64_t path_count,
                       upbp_light_paths& out);

}  // namespace upbp
