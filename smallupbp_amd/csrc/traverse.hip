// traverse.hip -- query traversal kernels for gfx950 (wave64).
//
// One wavefront carries a bundle of 64 query beams (one per lane). The wave
// walks ONE traversal of the LBVH: every node record is fetched once per wave
// from a wave-uniform address (scalar loads), each lane slab-tests its own ray
// segment against the two child boxes, and __ballot decides where the wave
// goes. Leaf items (photons or beam pieces) are also fetched once per wave and
// tested by every lane against its own ray. The traversal stack holds
// wave-uniform node indices, one entry per lane register (two VGPRs = 128
// entries), pushed with a lane-select and popped with readlane.
//
// Per query the segment loop of EmbreeBre::evalBre (SmallUPBP/src/Bre/Bre.cxx:812-879,
// lite :895-964) and PhotonBeamsEvaluator::evalBeamBeamEstimate
// (SmallUPBP/src/Beams/PhBeams.cxx:177-241, lite :257-324) runs in registers:
// result += P * segment_result, P *= attenuation (/ pdf for SHORT queries), stop
// when a channel of P is <= 1e-20. Per hit the plain callbacks are evaluated:
// breIntersectFuncHomogeneous (Bre.cxx:239-277) and PhotonBeam::accumulate
// (SmallUPBP/src/Beams/PhotonBeam.hxx:315-367). The adjoint mode re-traverses
// and recomputes transmittance per hit instead of storing it.
#include <algorithm>

#include "upbp_internal.hpp"
#include "upbp_mis.hpp"

namespace upbp {

namespace {

constexpr int kWave = 64;
constexpr int kStackMax = 128;
constexpr int kEstPhotons = 0, kEstBeams = 1;
constexpr int kMaxLdsMedia = 8;  // adjoint: per-lane medium gradient slabs held in LDS

struct EvalArgs {
    // structure
    const NodeDev* __restrict__ nodes;
    const float4* __restrict__ pos_r2;
    const float4* __restrict__ power;
    const float4* __restrict__ inc;
    const uint32_t* __restrict__ orig;  // photon original index / piece -> beam index
    const uint64_t* __restrict__ end_bits;  // a bit per piece: a beam's first or last (one more word after)
    const PieceDev* __restrict__ pieces;
    const float4* __restrict__ piece_flux;
    // queries
    const float* __restrict__ origin;
    const float* __restrict__ direction;
    const int64_t* __restrict__ offsets;
    const upbp_volume_segment* __restrict__ segments;
    const uint32_t* __restrict__ perm;
    int64_t count;
    int32_t short_query;
    int32_t lite;
    // media
    const MediumDev* __restrict__ media;
    int32_t n_media;
    int32_t media_base;
    int32_t lds_media_n;  // adjoint: media with an LDS gradient slab (min(n_media, kMaxLdsMedia))
    // outputs
    float* __restrict__ out;
    uint32_t* __restrict__ sig;
    unsigned long long* __restrict__ stats;
    // adjoint
    const float* __restrict__ grad_out;
    float* __restrict__ grad_media;  // [grad_mask + 1][M][6]: a wave adds to its block's row
    float* __restrict__ grad_items;  // [items][3]
    // UPBP mode
    const upbp_query_mis* __restrict__ qmis;
    MisGlobals mis;
    // traversal starts here (0, or an instance's root in a batched plan's merged tree array)
    uint32_t root;
    // a wave with a frustum tests an inner node's subtree of at most this many items as one leaf
    uint32_t frustum_leaf;
    // per-cell beam reduction of the beam estimators (red.max == 0: none)
    RedDev red;
    // split tiles: wave w gathers part w % 2^log_parts of tile w / 2^log_parts into row row0 + w, or does
    // tasks[w] (of plan->n_tasks; tile_task); a part's sums go to rows[row][3][64] (signatures: [2][64]),
    // which k_sum_rows adds up
    const uint2* __restrict__ tasks;
    PlanWords* __restrict__ plan;
    uint32_t shift;  // ItemPart::shift of one part; half the items per block for twice the parts, at least 64
    uint32_t log_parts, row0;
    uint32_t grad_mask;  // adjoint
    float* __restrict__ rows;
    // in_two: whether this launch's tiles are known (a plan's tasks; the tiles that tile_class gives, the
    // plan's costs, as kCostOther; or all); else each wave finds out by itself (common_origin)
    const uint32_t* __restrict__ tile_class;
    uint32_t known;
};
constexpr uint32_t kCostOther = 0xFFFFFFFFu;  // of a tile without an estimate, whose rays have no common origin

// The items a wave gathers: the blocks of 2^shift items of leaf order whose index is p modulo
// mask + 1. Blocks are dealt out in turn, because the items that one tile meets often lie close
// together in that order (the beams that leave one light).
struct ItemPart {
    uint32_t p, mask, shift;
    // whether some of the n items from s on are this part's
    __device__ __forceinline__ bool meets(uint32_t s, uint32_t n) const {
        const uint32_t b = s >> shift;
        return ((p - b) & mask) <= ((s + n - 1u) >> shift) - b;
    }
    // which of the n <= 64 items from s on are (they lie in at most two blocks, of 64 items or more)
    __device__ __forceinline__ uint64_t items(uint32_t s, uint32_t n) const {
        const uint64_t all = n >= 64u ? ~0ull : ((1ull << n) - 1ull);
        const uint32_t b = s >> shift, first = ((b + 1u) << shift) - s;  // items left in the first block
        const uint64_t low = first >= 64u ? ~0ull : ((1ull << first) - 1ull);
        const uint64_t mine = (((p - b) & mask) == 0u ? low : 0ull) | (((p - b - 1u) & mask) == 0u ? ~low : 0ull);
        return all & mine;
    }
};

// The work of wave w of a split launch.
struct TileTask {
    uint32_t tile, row, log_parts;
    ItemPart part;
};
constexpr uint32_t kTaskPartBits = 8, kTaskLogBits = 4;  // of a task's second word, then the row
__device__ __forceinline__ TileTask tile_task(const uint2* tasks, uint32_t log_parts, uint32_t row0, uint32_t shift,
                                              uint32_t w) {
    TileTask t;
    uint32_t p;
    if (tasks) {
        const uint2 v = tasks[w];
        t.tile = v.x;
        p = v.y & ((1u << kTaskPartBits) - 1u);
        t.log_parts = (v.y >> kTaskPartBits) & ((1u << kTaskLogBits) - 1u);
        t.row = v.y >> (kTaskPartBits + kTaskLogBits);
    } else {
        t.tile = w >> log_parts;
        p = w & ((1u << log_parts) - 1u);
        t.log_parts = log_parts;
        t.row = row0 + w;
    }
    t.part = {p, (1u << t.log_parts) - 1u, (uint32_t)max((int)shift - (int)t.log_parts, 6)};
    return t;
}

__device__ __forceinline__ float guard_inv(float d) {
    const float a = __builtin_fabsf(d) < 1e-20f ? __builtin_copysignf(1e-20f, d) : d;
    return __builtin_amdgcn_rcpf(a);
}

struct Ray {
    float ox, oy, oz, dx, dy, dz;
    float ix, iy, iz;     // guarded reciprocal direction
    float oix, oiy, oiz;  // o * inv
    float d1o1;           // dot3(d, o), loop invariant of the beam test
    uint64_t qkey;        // per-cell beam reduction: key of the query ray (reduced kernels only)
};

// Wave mask of the lanes whose segment [tmin, tmax] meets the box:
// max(tn, tmin) <= min(tf, tmax) as three compares, each balloted on its own. min / max of
// tmin and tmax (values the compiler cannot prove canonical) would put a canonicalising max
// in front of each use at every node, and a ballot of a combined bool first selects it into
// a VGPR and compares it back; the slab values are fma results and need neither.
__device__ __forceinline__ uint64_t slab_mask(const Ray& r, float tmin, float tmax, float lx, float ly, float lz,
                                              float hx, float hy, float hz) {
    const float ax = __builtin_fmaf(lx, r.ix, -r.oix), bx = __builtin_fmaf(hx, r.ix, -r.oix);
    const float ay = __builtin_fmaf(ly, r.iy, -r.oiy), by = __builtin_fmaf(hy, r.iy, -r.oiy);
    const float az = __builtin_fmaf(lz, r.iz, -r.oiz), bz = __builtin_fmaf(hz, r.iz, -r.oiz);
    const float tn = fmaxf(fmaxf(fminf(ax, bx), fminf(ay, by)), fminf(az, bz));
    const float tf = fminf(fminf(fmaxf(ax, bx), fmaxf(ay, by)), fmaxf(az, bz));
    return __ballot(tn <= tf) & __ballot(tn <= tmax) & __ballot(tf >= tmin);
}

__device__ __forceinline__ uint32_t uni(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// A wave-uniform global pointer read from memory, made a scalar: the two halves pass
// through readfirstlane and the result is tagged as global memory, so loads through it
// use a scalar base (as kernel-argument pointers do) instead of a 64-bit VGPR pair.
// 64-bit readfirstlane from two 32-bit halves. readfirstlane returns int: each half
// goes through uint32_t before widening, or a low word with bit 31 set would
// sign-extend over the high word.
__device__ __forceinline__ uint64_t uni_u64(uint64_t v) {
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)v);
    return ((uint64_t)hi << 32) | (uint64_t)lo;
}

// The kernel's arguments read again from memory (KARG: A is k_eval's only argument; else A itself), for
// the code around the traversal: values the compiler would otherwise load once and keep in scalar
// registers through the traversal loop, or spill into lanes of vector registers there. `after` is a
// scalar that the reads must wait for. (Not volatile: that would count as a write to memory, and the
// traversal's node and item reads would no longer be scalar loads.)
template <bool KARG, class Args>
__device__ __forceinline__ const Args* reread(const Args& A, uint32_t after) {
    if (!KARG) return &A;
    auto p = (const __attribute__((address_space(4))) Args*)(uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm("" : "+s"(p) : "s"(after));
    return (const Args*)p;
}

// A pointer to global memory, however it was read.
template <class T>
__device__ __forceinline__ T* as_global(T* p) {
    return (T*)(__attribute__((address_space(1))) T*)p;
}

template <class T>
__device__ __forceinline__ T* uni_global(T* p) {
    return (T*)(__attribute__((address_space(1))) T*)uni_u64((uint64_t)p);
}

__device__ __forceinline__ int64_t uni64(int64_t x) { return (int64_t)uni_u64((uint64_t)x); }

// Lane state of one segment being gathered.
struct SegState {
    float tmin, tmax;
    float x0, x1, x2;  // per channel, what a length of the query adds to log2 of its factor (set_factors)
    float ek;          // sigma_t log2(e) of the smallest sigma_t (what SHORT beams are normalised by)
    float ss0, ss1, ss2;
    float g;           // 0 for isotropic media, where phase_pdf gives the constant exactly
    int32_t kidx;      // the smallest sigma_t's channel (adjoint)
    int32_t medium;     // medium id (instance-local, for the beam medium test)
    float min_comp, mfp, cont;  // UPBP mode: min sigma_t component, mean free path, continuation
    float acc0, acc1, acc2;
    // adjoint per segment: w (upstream) * prefix, and accumulators
    float w0, w1, w2;
    float gs0, gs1, gs2;  // d/d sigma_s direct
    float gt0, gt1, gt2;  // d/d sigma_t
};

// A MODE of Forward or Signature with this bit set applies the per-cell beam reduction
// (a separate instantiation: the plain kernels keep their registers).
constexpr int kReduced = 8;
// With this bit a tile's items are split over several waves (the others keep their registers too).
constexpr int kSplit = 16;
// The plain modes evaluate the waves whose rays share their origin; with this bit (a launch of its own,
// since its registers would cost the others) they evaluate the other waves.
constexpr int kSparse = 32;
// With this bit (batched plans) nodes and items are read as constant memory (uniform_at).
constexpr int kBatch = 64;
// base[i] for an index that is the same for the whole wave, in one scalar load. The persistent batched
// kernel writes memory (its queue, its outputs) before it reads further nodes and items, so the compiler
// cannot know that they are never written and reads them with vector loads, a node in four that wait for
// one another; as constant memory they are known not to change while a kernel runs. 16 instances, 4.6M
// rays: 5.77 -> 4.60 ms; 16 instances x 30k rays without a common origin 6.80 -> 4.78 ms.
template <int MODE, class T>
__device__ __forceinline__ T uniform_at(const T* base, uint32_t i) {
    if (!(MODE & kBatch)) return base[i];
    static_assert(sizeof(T) % 16 == 0, "read in 16-byte words");
    typedef float Word __attribute__((ext_vector_type(4)));
    Word w[sizeof(T) / 16];
    const auto* p = (const __attribute__((address_space(4))) Word*)(uint64_t)(base + i);
    for (size_t k = 0; k < sizeof(T) / 16; ++k) w[k] = p[k];
    T v;
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

// Whether a mode comes in those two launches.
constexpr bool in_two(int mode) {
    return ((mode & 7) == (int)Mode::Forward || (mode & 7) == (int)Mode::Signature) && !(mode & kReduced);
}

template <int MODE>
struct LaneOut {
    uint32_t hits = 0;
    uint32_t sig_n = 0, sig_h = 0;
    uint32_t err = 0;
    bool aniso = false;       // whether some lane's medium of the segment is anisotropic (wave-uniform)
    MisLane ml;               // UPBP mode only
    uint32_t qh = 0, qt = 0;  // UPBP, kSparse: head and tail of the wave's queue (wave-uniform)
};

__device__ __forceinline__ float pick3(int k, float a, float b, float c) { return k == 0 ? a : (k == 1 ? b : c); }

__device__ __forceinline__ float wave_sum(float v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// v + DPP-moved v; lanes outside row_mask add 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_add(float v) {
    const int m = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROW_MASK, 0xF, false);
    return v + __int_as_float(m);
}

// Sum over the 64 lanes of a wave with DPP row operations (all lanes must be active).
// quad_perm(1,0,3,2) and (2,3,0,1) sum quads, row_ror 4 and 8 sum rows of 16,
// row_bcast15 / row_bcast31 carry row sums upward; lane 63 ends with the total.
__device__ __forceinline__ float wave_sum_dpp(float v) {
    v = dpp_add<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
    v = dpp_add<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
    v = dpp_add<0x124, 0xF>(v);  // row_ror:4
    v = dpp_add<0x128, 0xF>(v);  // row_ror:8
    v = dpp_add<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// ---- leaf visitors ---------------------------------------------------------
// A hit's transmittance factors, exp2 of an exponent per channel c: a length adds -e_c to it, e_c =
// sigma_t_c log2(e), or where it is SHORT, whose transmittance is divided by channel k's, e_k - e_c. That
// is formed before it is multiplied by the length, so that the factor of channel k (of all channels of a
// grey medium) is exactly 1 there, however thick the medium: e_k times the SHORT lengths, rounded, less
// e_c times all lengths was off by 5e-6 of it at sigma_t 80 (and two instructions per beam hit less: 8.55
// instead of 8.64 ms for 1920x1080 rays x 1M photons + 200k SHORT beams). Three multiplies for a photon
// hit, three instructions per channel for a beam hit, and one exp2 each: the exponents with products,
// differences and selections per lane, and the per-lane choice of phase function, were 50 of the 80
// vector instructions of a beam hit and made that evaluation 11.8 ms; 10.9 ms without those and with the
// record read in one go (test_beam_beam).
struct Trans {
    float c0, c1, c2;
};
__device__ __forceinline__ void set_factors(SegState& s, float st0, float st1, float st2, int min_idx, bool short_q) {
    const float stk = pick3(min_idx, st0, st1, st2);
    s.ek = stk * kLog2e;
    s.x0 = (short_q ? stk - st0 : -st0) * kLog2e;
    s.x1 = (short_q ? stk - st1 : -st1) * kLog2e;
    s.x2 = (short_q ? stk - st2 : -st2) * kLog2e;
}
// of a photon at dt along the query
__device__ __forceinline__ Trans transmittance(const SegState& s, float dt) {
    return {__builtin_amdgcn_exp2f(s.x0 * dt), __builtin_amdgcn_exp2f(s.x1 * dt), __builtin_amdgcn_exp2f(s.x2 * dt)};
}
// of dq along the query and t2 along a beam; kb: 1 for a SHORT beam less 1 for a SHORT query (short_diff)
__device__ __forceinline__ float short_diff(bool short_b, bool short_q) {
    return (short_b ? 1.f : 0.f) - (short_q ? 1.f : 0.f);
}
__device__ __forceinline__ Trans transmittance(const SegState& s, float dq, float t2, float kb) {
    return {__builtin_amdgcn_exp2f(__builtin_fmaf(__builtin_fmaf(kb, s.ek, s.x0), t2, s.x0 * dq)),
            __builtin_amdgcn_exp2f(__builtin_fmaf(__builtin_fmaf(kb, s.ek, s.x1), t2, s.x1 * dq)),
            __builtin_amdgcn_exp2f(__builtin_fmaf(__builtin_fmaf(kb, s.ek, s.x2), t2, s.x2 * dq))};
}

// Sums the three channels' item gradients over the wave (DPP) and adds them once: lanes 0 to 2 add one
// channel each in one instruction, to neighbouring words (512x512 forward and adjoint: 10.6 ms with one
// lane adding all three, 10.0 ms).
__device__ __forceinline__ void add_item_gradient(float* grad, uint32_t o, float g0, float g1, float g2) {
    const float r0 = wave_sum_dpp(g0), r1 = wave_sum_dpp(g1), r2 = wave_sum_dpp(g2);
    const int lane = threadIdx.x & (kWave - 1);
    if (lane < 3) unsafeAtomicAdd(&grad[3 * o + lane], lane == 0 ? r0 : lane == 1 ? r1 : r2);
}

__device__ __forceinline__ MisF merge_vertex_mis(const upbp_mis_params& P, float pdf_a_inv, float ray_pdf_inv,
                                                 float ratio, float bb1d_sel, uint32_t flags) {
    MisF m = {};
    m.pdf_a_inv = pdf_a_inv;
    m.ray_sample_pdf_inv = ray_pdf_inv;
    m.ray_sample_pdfs_ratio = ratio;
    m.surf = 0.f;
    m.pp3d = P.pp3d_factor;
    m.pb2d = P.pb2d_factor;
    m.bb1d = P.bb1d_factor;
    m.bb1d_sel = bb1d_sel;
    m.flags = flags;
    return m;
}

// breIntersectFuncHomogeneous2 after the disc test (Bre.cxx:305-463), per lane; the
// photon's light vertex is read by index (lanes hit different photons only through
// the same wave-uniform photon, so this is one gather per hit).
__device__ void photon_hit_mis(const EvalArgs& A, const Ray& r, SegState& s, const MisLane& ml, float t, float sq,
                               float r2, uint32_t lv_idx, bool short_q, uint32_t& err) {
    const MisGlobals& G = A.mis;
    const upbp_mis_params& P = G.p;
    if ((int64_t)lv_idx >= G.lv_count) {
        err |= kBadLightIndex;
        return;
    }
    // the vertex's record: its fields, and those of the walk's index 1 with its tail, in one read
    const PhotonRec rec = G.photon_recs[lv_idx];
    const uint32_t path_len = rec.d.x & kRecLengthMask;
    const uint32_t cam_len = (uint32_t)ml.cam_len;
    if ((path_len + cam_len > P.max_path_length) || (path_len + cam_len < P.min_path_length)) return;
    if (cam_len == 1 && t < P.min_dist_to_med) return;
    // The weights and contributions below need 1e-4 relative accuracy, not the reference's
    // rounding (hit decisions are all made before this point), so reciprocals and square
    // roots are the single hardware instructions.
    const float dt = t - s.tmin;
    const float pdf = __builtin_amdgcn_exp2f(-s.ek * dt);
    const Trans tr = transmittance(s, dt);
    const float a0 = tr.c0, a1 = tr.c1, a2 = tr.c2;
    float ray_pdf = s.min_comp * pdf;
    float ray_rev = (ml.seg_flags & UPBP_ORIGIN_IN_MEDIUM) ? ray_pdf : pdf;
    const float ratio = __builtin_amdgcn_rcpf(s.min_comp);
    if (!(a0 > 1e-20f && a1 > 1e-20f && a2 > 1e-20f)) return;
    ray_pdf *= ml.pref_pdf;
    ray_rev *= ml.pref_rev;
    // PhaseFunction::Evaluate(-ray.dir, lightDirection): cos = -dot(gen, fix) = dot(dir_fix, d)
    const float lx = rec.b.x, ly = rec.b.y, lz = rec.b.z;
    const float cos_t = -dot3(lx, ly, lz, -r.dx, -r.dy, -r.dz);
    const float bsdf = phase_pdf(s.g, false, cos_t);
    const float sin_t = __builtin_amdgcn_sqrtf(fmaxf(0.f, 1.f - cos_t * cos_t));
    if (bsdf <= 0.f) return;
    const float dir_pdf = bsdf * s.cont;
    const float rev_pdf = bsdf * rec.a.w;
    const float kernel = radial_kernel(sq, r2) * __builtin_amdgcn_rcpf((r2 * kPi) * 0.5f);
    if (!(kernel > 1e-20f)) return;
    const float u0 = (((rec.a.x * a0) * s.ss0) * bsdf) * kernel;
    const float u1 = (((rec.a.y * a1) * s.ss1) * bsdf) * kernel;
    const float u2 = (((rec.a.z * a2) * s.ss2) * bsdf) * kernel;
    if (u0 <= 0.f && u1 <= 0.f && u2 <= 0.f) return;
    const float dist_sq = t * t;
    const float ray_pdf_inv = __builtin_amdgcn_rcpf(ray_pdf);
    // Bre.cxx:407-415: the photon-beam evaluator's getBeamSelectionPdf(isectPt) when it reduces
    // its cells (A.red is then its grid), 1 when it does not, 0 without photon beams
    float sel = P.has_bb1d_beams ? 1.f : 0.f;
    if (P.has_bb1d_beams && A.red.max) sel = red_cell_pdf(A.red, r.ox + t * r.dx, r.oy + t * r.dy, r.oz + t * r.dz);
    const MisF mv = merge_vertex_mis(P, ml.last_pdf_w_inv * dist_sq * ray_pdf_inv, ray_pdf_inv, ratio, sel,
                                     s.mfp > P.bb1d_min_mfp ? UPBP_MIS_IN_MEDIUM_WITH_BEAMS : 0u);
    const float last = short_q ? __builtin_amdgcn_rcpf(ratio * mv.pb2d) : ray_pdf * __builtin_amdgcn_rcpf(mv.pb2d);
    const uint32_t tech = A.short_query ? (UPBP_SHORT_BEAM | P.techniques) : (UPBP_LONG_BEAM | P.techniques);
    const float w_cam = camera_weight_tail(ml.tail, mv, last, sin_t, rec.b.w, rec.c.x,
                                           rev_pdf * ray_rev * __builtin_amdgcn_rcpf(dist_sq),
                                           __builtin_amdgcn_rcpf(ray_rev), P.query_beam_type, P.photon_beam_type,
                                           tech);
    float w_light;
    if (!light_weight_tail_prec(rec, last, dir_pdf, tech, w_light)) {
        LightView lview{&G, nullptr, -1, 0.f};
        w_light = light_path_weight(lview, (int)rec.d.y, (int)path_len, last, dir_pdf, UPBP_PB2D, P.query_beam_type,
                                    P.photon_beam_type, tech, err);
    }
    const float w = __builtin_amdgcn_rcpf(w_light + w_cam);
    s.acc0 += w * u0;
    s.acc1 += w * u1;
    s.acc2 += w * u2;
}

// PhotonBeam::accumulate2 after the beam-beam test (PhotonBeam.hxx:393-605). The beam,
// its MIS record and its origin light vertex are wave-uniform (scalar loads).
// sel_pdf: the beam selection pdf of the hit's reduction cell (1 without reduction); mult: the
// times that cell tests the beam, each test adding the weighted contribution.
__device__ void beam_hit_mis(const EvalArgs& A, const Ray& r, SegState& s, const MisLane& ml, float dist,
                             float sin_theta, float t1, float t2, float radius, bool short_b, float4 flux,
                             float d2x, float d2y, float d2z, uint32_t beam_idx, float sel_pdf, uint32_t mult,
                             bool short_q, uint32_t& err) {
    const MisGlobals& G = A.mis;
    const upbp_mis_params& P = G.p;
    // the beam's record: its MIS fields, origin light vertex and light tail in one 64-byte read
    const BeamRec rec = G.beam_recs[beam_idx];
    if (rec.info & kRecBadVertex) {
        err |= kBadLightIndex;
        return;
    }
    const uint32_t path_len = rec.info & kRecLengthMask;
    const uint32_t cam_len = (uint32_t)ml.cam_len;
    if ((path_len + 1 + cam_len > P.max_path_length) || (path_len + 1 + cam_len < P.min_path_length)) return;
    if (cam_len == 1 && t1 < P.min_dist_to_med) return;
    // As in photon_hit_mis, everything below is weight and contribution arithmetic with a
    // 1e-4 budget: hardware reciprocals, and one exponential per channel for the query and
    // beam transmittances together (with the SHORT normalisations folded into the exponent).
    const float dq = t1 - s.tmin;
    const float pq = __builtin_amdgcn_exp2f(-s.ek * dq), pb = __builtin_amdgcn_exp2f(-s.ek * t2);
    const Trans tr = transmittance(s, dq, t2, short_diff(short_b, short_q));
    const float a0 = tr.c0, a1 = tr.c1, a2 = tr.c2;
    float rsp_q = s.min_comp * pq;
    float rsr_q = (ml.seg_flags & UPBP_ORIGIN_IN_MEDIUM) ? rsp_q : pq;
    float rsp_b = s.min_comp * pb;
    float rsr_b = (rec.info & kRecOriginInMedium) ? rsp_b : pb;
    const float ratio = __builtin_amdgcn_rcpf(s.min_comp);  // ratio_q = ratio_b
    if (!(a0 > 1e-20f && a1 > 1e-20f && a2 > 1e-20f)) return;
    rsp_q *= ml.pref_pdf;
    rsr_q *= ml.pref_rev;
    rsp_b *= rec.ray_sample_pdf;
    rsr_b *= rec.ray_sample_rev_pdf;
    // PhaseFunction::Evaluate(-ray.direction, -beam.direction): cos = -dot(-d2, -d1)
    const float cos_t = -dot3(-d2x, -d2y, -d2z, -r.dx, -r.dy, -r.dz);
    const float bsdf = phase_pdf(s.g, false, cos_t);
    if (bsdf <= 0.f) return;
    const float dir_pdf = bsdf * s.cont;
    const float rev_pdf = bsdf * s.cont;
    // 1D kernel (1 - dist^2/r^2) * 3 / (4 r sin(theta)) / selection pdf (PhotonBeam.hxx:487-494)
    const float k1 = radial_kernel(dist * dist, radius * radius) * 3.0f;
    const float kd = k1 * __builtin_amdgcn_rcpf((4.0f * radius) * sin_theta) * __builtin_amdgcn_rcpf(sel_pdf);
    const float u0 = ((((flux.x * s.ss0) * a0) * bsdf) * kd);
    const float u1 = ((((flux.y * s.ss1) * a1) * bsdf) * kd);
    const float u2 = ((((flux.z * s.ss2) * a2) * bsdf) * kd);
    if (u0 <= 0.f && u1 <= 0.f && u2 <= 0.f) return;
    const float dist_sq_q = t1 * t1;
    const float rsp_inv_q = __builtin_amdgcn_rcpf(rsp_q);
    const MisF mv = merge_vertex_mis(P, ml.last_pdf_w_inv * dist_sq_q * rsp_inv_q, rsp_inv_q, ratio, sel_pdf,
                                     UPBP_MIS_IN_MEDIUM_WITH_BEAMS);
    const float dist_sq_b = (rec.info & kRecFinite) ? t2 * t2 : 1.0f;
    const float rsp_inv_b = __builtin_amdgcn_rcpf(rsp_b);
    const MisF bv = merge_vertex_mis(P, rec.last_pdf_w_inv * dist_sq_b * rsp_inv_b, rsp_inv_b, ratio, sel_pdf,
                                     UPBP_MIS_IN_MEDIUM_WITH_BEAMS);
    const uint32_t tech = A.short_query ? (UPBP_SHORT_BEAM | P.techniques) : (UPBP_LONG_BEAM | P.techniques);
    const float sin_t = (tech & UPBP_NO_SINE_IN_WEIGHTS) ? 1.0f : sin_theta;
    // PhotonBeam.hxx:555-564: 1 / (the merged technique's pdf) per beam-type pair
    const float tp = mv.bb1d * sel_pdf * sin_t;
    float last;
    if (short_q)
        last = short_b ? __builtin_amdgcn_rcpf(ratio * ratio * tp) : rsp_b * __builtin_amdgcn_rcpf(ratio * tp);
    else
        last = short_b ? rsp_q * __builtin_amdgcn_rcpf(ratio * tp) : rsp_q * rsp_b * __builtin_amdgcn_rcpf(tp);
    const float w_cam = camera_weight_tail(ml.tail, mv, last, sin_t, rsp_inv_b, ratio,
                                           rev_pdf * rsr_q * __builtin_amdgcn_rcpf(dist_sq_q),
                                           __builtin_amdgcn_rcpf(rsr_q), P.query_beam_type, P.photon_beam_type, tech);
    const uint32_t lvf = rec.lv_flags;
    const bool on_light_delta = (lvf & UPBP_MIS_ON_LIGHT_SOURCE) && (lvf & UPBP_MIS_DELTA);
    const float ntl = on_light_delta
                          ? 0.f
                          : dir_pdf * rsr_b * __builtin_fabsf(rec.cos_theta_out) * __builtin_amdgcn_rcpf(dist_sq_b);
    const float rsr_inv_b = __builtin_amdgcn_rcpf(rsr_b);
    float w_light;
    if (!light_weight_tail_rec(rec, last, bv.pdf_a_inv, ntl, rsr_inv_b, tech, w_light)) {
        LightView lview{&G, &bv, (int64_t)rec.light_vertex, rsr_inv_b};
        w_light = light_path_weight(lview, rec.path_idx, (int)path_len + 1, last, ntl, UPBP_BB1D, P.query_beam_type,
                                    P.photon_beam_type, tech, err);
    }
    const float w = __builtin_amdgcn_rcpf(w_light + w_cam) * (float)mult;
    s.acc0 += w * u0;
    s.acc1 += w * u1;
    s.acc2 += w * u2;
}

// ---- UPBP hit queue ----------------------------------------------------------
// A hit's MIS weight costs a few hundred instructions, and when a wave tests an item only
// about 20 of its 64 lanes hit it (21.5 photon and 18.2 beam hits per item with any hit,
// 1920x1080 UPBP workload). Evaluated in place, the weight would run with two thirds of
// the lanes idle. So each wave queues its hits in LDS and evaluates them 64 at a time:
// a lane takes one queued hit, reads the owner lane's ray, segment and camera state with
// ds_bpermute, and the weighted contribution goes back to the owner's LDS accumulator
// with a float atomic. The queue drains completely before the segment ends, because the
// owner's segment state is what the weights read.
constexpr int kHq = 128;     // ring entries per wave: a ballot adds at most 64 to fewer than 64 queued
constexpr int kHqWaves = 4;  // waves per block of the UPBP launches (launch_mode clamps to 4)
constexpr int kHqWords = 7;  // words per queued hit
// Some lanes write g_hq, g_pq and g_hacc and others read them: through lds_read and lds_write. (With
// wave_lds_sync around the evaluations the traversal's node and item reads are no longer scalar loads:
// weighted 1920x1080 rays took 20.5 instead of 19.1 ms, 200k rays without a common origin 18.4 instead of
// 14.9 ms.)
__shared__ uint32_t g_hq[kHqWaves][kHqWords][kHq];
__shared__ float g_hacc[kHqWaves][3][kWave];

// Position of this lane's entry among the set bits of m below it.
__device__ __forceinline__ uint32_t lane_rank(uint64_t m) {
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

__device__ __forceinline__ float from_lane(float v, int src) { return __shfl(v, src, kWave); }
__device__ __forceinline__ int32_t from_lane(int32_t v, int src) { return __shfl(v, src, kWave); }
__device__ __forceinline__ uint32_t from_lane(uint32_t v, int src) { return (uint32_t)__shfl((int)v, src, kWave); }

// The owner lane's state that photon_hit_mis / beam_hit_mis read (all lanes take part).
__device__ __forceinline__ void owner_state(const Ray& r, const SegState& s, const MisLane& ml, int owner, Ray& ro,
                                            SegState& so, MisLane& mo) {
    ro.dx = from_lane(r.dx, owner);
    ro.dy = from_lane(r.dy, owner);
    ro.dz = from_lane(r.dz, owner);
    so.tmin = from_lane(s.tmin, owner);
    so.x0 = from_lane(s.x0, owner);
    so.x1 = from_lane(s.x1, owner);
    so.x2 = from_lane(s.x2, owner);
    so.ek = from_lane(s.ek, owner);
    so.ss0 = from_lane(s.ss0, owner);
    so.ss1 = from_lane(s.ss1, owner);
    so.ss2 = from_lane(s.ss2, owner);
    so.g = from_lane(s.g, owner);
    so.min_comp = from_lane(s.min_comp, owner);
    so.mfp = from_lane(s.mfp, owner);
    so.cont = from_lane(s.cont, owner);
    so.acc0 = so.acc1 = so.acc2 = 0.f;
    mo.tail.c = from_lane(ml.tail.c, owner);
    mo.tail.co = from_lane(ml.tail.co, owner);
    mo.tail.fl = from_lane(ml.tail.fl, owner);
    mo.cam_len = from_lane(ml.cam_len, owner);
    mo.last_pdf_w_inv = from_lane(ml.last_pdf_w_inv, owner);
    mo.pref_pdf = from_lane(ml.pref_pdf, owner);
    mo.pref_rev = from_lane(ml.pref_rev, owner);
    mo.seg_flags = from_lane(ml.seg_flags, owner);
}

__device__ __forceinline__ void return_to_owner(int w, int owner, const SegState& so) {
    atomicAdd(&g_hacc[w][0][owner], so.acc0);
    atomicAdd(&g_hacc[w][1][owner], so.acc1);
    atomicAdd(&g_hacc[w][2][owner], so.acc2);
}

// Evaluates the first n (1..64) queued photon hits: [0] light vertex, [1] owner lane,
// [2] t, [3] squared distance, [4] r^2.
template <int MODE>
__device__ __forceinline__ void drain_photons(const EvalArgs& A, const Ray& r, const SegState& s,
                                              LaneOut<MODE>& lo, uint32_t n, bool short_q) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const uint32_t pos = (lo.qh + (uint32_t)lane) & (kHq - 1);
    const bool act = (uint32_t)lane < n;
    const int owner = act ? (int)(lds_read(g_hq[w][1][pos]) & (kWave - 1)) : lane;
    Ray ro = {};
    SegState so;
    MisLane mo;
    owner_state(r, s, lo.ml, owner, ro, so, mo);
    if (A.red.max) {  // the hit point's reduction cell needs the owner's origin (wave-uniform branch)
        ro.ox = from_lane(r.ox, owner);
        ro.oy = from_lane(r.oy, owner);
        ro.oz = from_lane(r.oz, owner);
    }
    if (act) {
        photon_hit_mis(A, ro, so, mo, __uint_as_float(lds_read(g_hq[w][2][pos])), __uint_as_float(lds_read(g_hq[w][3][pos])),
                       __uint_as_float(lds_read(g_hq[w][4][pos])), lds_read(g_hq[w][0][pos]), short_q, lo.err);
        return_to_owner(w, owner, so);
    }
    lo.qh += n;
}

// The same for beam hits: [0] piece, [1] owner lane | SHORT beam << 8 | times counted << 9,
// [2] dist, [3] sin(theta), [4] t1, [5] t2, [6] radius (reduced kernels: the cell's selection
// pdf; the radius r0 + t2 dr is then recomputed from the piece, the same operations as the
// beam test's).
template <int MODE>
__device__ __forceinline__ void drain_beams(const EvalArgs& A, const Ray& r, const SegState& s, LaneOut<MODE>& lo,
                                            uint32_t n, bool short_q) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const uint32_t pos = (lo.qh + (uint32_t)lane) & (kHq - 1);
    const bool act = (uint32_t)lane < n;
    const uint32_t meta = lds_read(g_hq[w][1][pos]);
    const int owner = act ? (int)(meta & (kWave - 1)) : lane;
    Ray ro = {};
    SegState so;
    MisLane mo;
    owner_state(r, s, lo.ml, owner, ro, so, mo);
    if (act) {
        const uint32_t i = lds_read(g_hq[w][0][pos]);
        const float4 d2 = A.pieces[i].p1;
        const float t2 = __uint_as_float(lds_read(g_hq[w][5][pos]));
        const float w6 = __uint_as_float(lds_read(g_hq[w][6][pos]));
        float radius = w6, sel_pdf = 1.0f;
        if (MODE & kReduced) {
            radius = d2.w + t2 * A.pieces[i].p3.y;
            sel_pdf = w6;
        }
        beam_hit_mis(A, ro, so, mo, __uint_as_float(lds_read(g_hq[w][2][pos])), __uint_as_float(lds_read(g_hq[w][3][pos])),
                     __uint_as_float(lds_read(g_hq[w][4][pos])), t2, radius, ((meta >> 8) & 1u) != 0u, A.piece_flux[i], d2.x,
                     d2.y, d2.z, A.orig[i], sel_pdf, meta >> 9, short_q, lo.err);
        return_to_owner(w, owner, so);
    }
    lo.qh += n;
}

// End of a segment: evaluates what is still queued and moves the owners' sums into s.acc.
template <int EST, int MODE>
__device__ __forceinline__ void upbp_segment_end(const EvalArgs& A, const Ray& r, SegState& s, LaneOut<MODE>& lo,
                                                 bool short_q) {
    const uint32_t n = uni(lo.qt - lo.qh);
    if (n) {
        if (EST == kEstPhotons)
            drain_photons<MODE>(A, r, s, lo, n, short_q);
        else
            drain_beams<MODE>(A, r, s, lo, n, short_q);
    }
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    s.acc0 += lds_read(g_hacc[w][0][lane]);
    s.acc1 += lds_read(g_hacc[w][1][lane]);
    s.acc2 += lds_read(g_hacc[w][2][lane]);
    lds_write(g_hacc[w][0][lane], 0.f);
    lds_write(g_hacc[w][1][lane], 0.f);
    lds_write(g_hacc[w][2][lane], 0.f);
}

// Tests the photons start + j of a leaf for the bits j of items (ascending).
template <int MODE>
__device__ __forceinline__ void photon_leaf(const EvalArgs& A, const Ray& r, SegState& s, LaneOut<MODE>& lo,
                                            uint32_t start, uint64_t items, bool short_q) {
    while (items) {
        const uint32_t i = start + (uint32_t)__builtin_ctzll(items);
        items &= items - 1;
        const float4 p = uniform_at<MODE>(A.pos_r2, i);  // scalar load, wave-uniform index
        float t, sq;
        const bool hit = test_bre(r.ox, r.oy, r.oz, r.dx, r.dy, r.dz, s.tmin, s.tmax, p.x, p.y, p.z, p.w, t, sq);
        if ((MODE & 7) == (int)Mode::Upbp) {
            const uint64_t m = __ballot(hit);
            if (m) {
                const uint32_t lv_idx = A.orig[i];
                if (hit) {
                    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
                    const uint32_t pos = (lo.qt + lane_rank(m)) & (kHq - 1);
                    lds_write(g_hq[w][0][pos], lv_idx);
                    lds_write(g_hq[w][1][pos], (uint32_t)lane);
                    lds_write(g_hq[w][2][pos], __float_as_uint(t));
                    lds_write(g_hq[w][3][pos], __float_as_uint(sq));
                    lds_write(g_hq[w][4][pos], __float_as_uint(p.w));
                    lo.hits++;
                }
                lo.qt = uni(lo.qt + (uint32_t)__popcll(m));
                if (lo.qt - lo.qh >= (uint32_t)kWave) drain_photons<MODE>(A, r, s, lo, kWave, short_q);
            }
            continue;
        }
        // as in beam_leaf: only the adjoint needs the whole wave inside
        if ((MODE & 7) == (int)Mode::Adjoint ? __ballot(hit) != 0 : hit) {
            const float4 w = uniform_at<MODE>(A.power, i);  // (rgb, 1 / (r^2 pi / 2))
            float gp0 = 0.f, gp1 = 0.f, gp2 = 0.f;
            if (hit) {
                const float dt = t - s.tmin;
                const Trans tr = transmittance(s, dt);
                const float a0 = tr.c0, a1 = tr.c1, a2 = tr.c2;
                float ph = kInvPi * 0.25f;
                if (lo.aniso) {
                    const float4 in = uniform_at<MODE>(A.inc, i);
                    ph = phase_pdf(s.g, false, dot3(in.x, in.y, in.z, r.dx, r.dy, r.dz));
                }
                // Epanechnikov kernel (1 - s/r^2) / (r^2 pi / 2), Bre.cxx:272-273; the hardware
                // reciprocal except near the radius (radial_kernel)
                const float kern = radial_kernel(sq, p.w);
                const float scale = (ph * kern) * w.w;
                // base_c = a_c * scale; contribution_c = power_c * base_c * sigma_s_c
                const float b0 = a0 * scale, b1 = a1 * scale, b2 = a2 * scale;
                const float c0 = w.x * b0 * s.ss0, c1 = w.y * b1 * s.ss1, c2 = w.z * b2 * s.ss2;
                if ((MODE & 7) == (int)Mode::Adjoint) {
                    // s.w = dL/dout * P (prefix transmittance of earlier segments)
                    gp0 = s.w0 * b0 * s.ss0;
                    gp1 = s.w1 * b1 * s.ss1;
                    gp2 = s.w2 * b2 * s.ss2;
                    s.gs0 += s.w0 * b0 * w.x;
                    s.gs1 += s.w1 * b1 * w.y;
                    s.gs2 += s.w2 * b2 * w.z;
                    s.gt0 -= s.w0 * c0 * dt;
                    s.gt1 -= s.w1 * c1 * dt;
                    s.gt2 -= s.w2 * c2 * dt;
                    // SHORT query: T_c / T_k, so channel k gains +dt from every channel
                    if (short_q) {
                        const float sum = (s.w0 * c0 + s.w1 * c1) + s.w2 * c2;
                        if (s.kidx == 0) s.gt0 += sum * dt;
                        else if (s.kidx == 1) s.gt1 += sum * dt;
                        else s.gt2 += sum * dt;
                    }
                    s.acc0 += s.w0 * c0;
                    s.acc1 += s.w1 * c1;
                    s.acc2 += s.w2 * c2;
                } else {
                    s.acc0 += c0;
                    s.acc1 += c1;
                    s.acc2 += c2;
                }
                lo.hits++;
                if ((MODE & 7) == (int)Mode::Signature) {
                    lo.sig_n++;
                    lo.sig_h += hash32(A.orig[i]);
                }
            }
            if ((MODE & 7) == (int)Mode::Adjoint) add_item_gradient(A.grad_items, A.orig[i], gp0, gp1, gp2);
        }
    }
}

// ---- wave frustum of rays from one point ------------------------------------
// When every active lane of a wave starts its ray at the same point (the camera rays of a
// frame), four planes through that point bound the rays' directions, and every ray lies on
// the inner side of each. A photon lying beyond one of the planes by more than its radius, or a
// beam piece whose segment does (widened by its box margin), is then farther than its radius
// from every ray of the wave: no lane can accept it, and its test is skipped for the whole
// wave. One lane per item of a leaf does that check, so a leaf costs one pass however many
// items it holds (which is why such a wave also takes small subtrees as one leaf). The planes
// are wave-uniform and live in SGPRs (VGPRs are what limits the beam kernel's occupancy); the
// vector instructions of the check take them as scalar operands.
struct Frustum {
    float n[4][3];     // inner unit normals
    float ox, oy, oz;  // the common origin
    float om;          // the origin's part of the items' rounding margin: 1e-6 |o|_1
    float mx, my, mz;  // mean direction
    float spread;      // largest distance of a ray's direction from it
};

__device__ __forceinline__ float uni_f(float v) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

__device__ __forceinline__ float wave_min(float v) {
    for (int off = 32; off > 0; off >>= 1) v = fminf(v, __shfl_xor(v, off, kWave));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, kWave));
    return v;
}

// Builds the wave's frustum for the lanes with a segment (s.tmin <= s.tmax); false (no
// culling) when their origins differ or their directions spread over more than 60 degrees
// from the mean. The bounds of the direction slopes are widened by 1e-5 relative, far above
// their rounding, so every ray stays inside its planes.
__device__ bool make_frustum(const Ray& r, const SegState& s, Frustum& F) {
    const bool act = s.tmin <= s.tmax;
    const uint64_t am = __ballot(act);
    if (am == 0) return false;
    if (__ballot(act && !(s.tmin >= 0.f)) != 0) return false;  // hits only at t >= 0 lie inside
    const int fl = __builtin_ctzll(am);
    const float ox = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.ox), fl));
    const float oy = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.oy), fl));
    const float oz = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(r.oz), fl));
    if (__ballot(act && !(r.ox == ox && r.oy == oy && r.oz == oz)) != 0) return false;
    const float sx = wave_sum_dpp(act ? r.dx : 0.f), sy = wave_sum_dpp(act ? r.dy : 0.f),
                sz = wave_sum_dpp(act ? r.dz : 0.f);
    const float sn = __builtin_sqrtf((sx * sx + sy * sy) + sz * sz);
    if (!(sn > 0.f)) return false;
    const float mx = sx / sn, my = sy / sn, mz = sz / sn;  // mean direction
    const float dd = act ? (r.dx * mx + r.dy * my) + r.dz * mz : 1.f;
    if (__ballot(act && !(dd > 0.5f)) != 0) return false;
    const float sdx = r.dx - mx, sdy = r.dy - my, sdz = r.dz - mz;
    F.mx = uni_f(mx), F.my = uni_f(my), F.mz = uni_f(mz);
    F.spread = uni_f(wave_max(act ? __builtin_sqrtf((sdx * sdx + sdy * sdy) + sdz * sdz) : 0.f) * 1.0001f + 1e-6f);
    // U across the mean direction (crossed with the axis it has the least of), V = M x U
    const float amx = __builtin_fabsf(mx), amy = __builtin_fabsf(my), amz = __builtin_fabsf(mz);
    float ux, uy, uz;
    if (amx <= amy && amx <= amz) {
        ux = 0.f, uy = mz, uz = -my;  // M x (1,0,0)
    } else if (amy <= amz) {
        ux = -mz, uy = 0.f, uz = mx;  // M x (0,1,0)
    } else {
        ux = my, uy = -mx, uz = 0.f;  // M x (0,0,1)
    }
    const float un = __builtin_sqrtf((ux * ux + uy * uy) + uz * uz);
    ux /= un, uy /= un, uz /= un;
    const float vx = my * uz - mz * uy, vy = mz * ux - mx * uz, vz = mx * uy - my * ux;
    const float u = act ? ((r.dx * ux + r.dy * uy) + r.dz * uz) / dd : 0.f;
    const float v = act ? ((r.dx * vx + r.dy * vy) + r.dz * vz) / dd : 0.f;
    float u0 = wave_min(act ? u : INFINITY), u1 = wave_max(act ? u : -INFINITY);
    float v0 = wave_min(act ? v : INFINITY), v1 = wave_max(act ? v : -INFINITY);
    u0 -= 1e-5f * (1.f + __builtin_fabsf(u0));
    u1 += 1e-5f * (1.f + __builtin_fabsf(u1));
    v0 -= 1e-5f * (1.f + __builtin_fabsf(v0));
    v1 += 1e-5f * (1.f + __builtin_fabsf(v1));
    // inner normals: d.n >= 0 for every ray direction d inside the slope bounds
    float n[4][3] = {{ux - u0 * mx, uy - u0 * my, uz - u0 * mz},
                     {u1 * mx - ux, u1 * my - uy, u1 * mz - uz},
                     {vx - v0 * mx, vy - v0 * my, vz - v0 * mz},
                     {v1 * mx - vx, v1 * my - vy, v1 * mz - vz}};
    // every lane holds the same values (wave reductions of the same inputs): take lane 0's
    for (int k = 0; k < 4; ++k) {
        const float nn = __builtin_sqrtf((n[k][0] * n[k][0] + n[k][1] * n[k][1]) + n[k][2] * n[k][2]);
        F.n[k][0] = uni_f(n[k][0] / nn);
        F.n[k][1] = uni_f(n[k][1] / nn);
        F.n[k][2] = uni_f(n[k][2] / nn);
    }
    F.ox = ox, F.oy = oy, F.oz = oz;
    F.om = uni_f(1e-6f * ((__builtin_fabsf(ox) + __builtin_fabsf(oy)) + __builtin_fabsf(oz)));
    return true;
}

// The pieces [start, start + cnt) of a leaf that some ray of the wave may accept: lane j checks
// piece start + j against the wave's frustum. An inner piece owns only pairs whose closest
// point on the beam line lies on its own segment, and that point is within the beam's radius
// of a ray, so the segment widened by 1.01 of the largest radius (the piece box's margin)
// cannot lie beyond a plane. The first and last piece of a beam also own the pairs whose
// closest point tw lies beyond the beam's ends, which the reference accepts only when the
// rounding of its t2 lands inside. With S the coordinates involved, t2 and tw differ by at most
// about 2e-6 S / |q|, q the cosine between the two directions. So an end piece is checked as
// its segment lengthened by ext = 1.01 r beyond the beam's end, except where some ray of the wave
// may have |q| <= 8e-6 S / ext (four times that bound): there it is always kept, and culling drops
// no pair that the visited leaf (or subtree) boxes reach. Always keeping every end piece made
// them 45 % of the pieces tested on 1920x1080 rays x 1M photons + 200k SHORT beams (32.8 of 73.0
// million, a quarter of them with any ray within the radius of the beam's line): the evaluation
// took 12.76 ms, now 11.37 ms; 1M rays x 2M beams 62.8 -> 59.2 ms; UPBP 23.6 -> 22.0 ms.
__device__ __forceinline__ uint64_t frustum_items(const EvalArgs& A, const Frustum& F, uint32_t start,
                                                  uint32_t cnt) {
    const int lane = threadIdx.x & (kWave - 1);
    bool out = false;
    if ((uint32_t)lane < cnt) {
        const float4 p0 = A.pieces[start + lane].p0, p1 = A.pieces[start + lane].p1,
                     p2 = A.pieces[start + lane].p2;
        // A margin only, so the hardware square root (within 1 ulp) does, and the plane
        // distances are fused multiply-adds: the 1e-6 relative margin is far above the error.
        const float rb = __builtin_amdgcn_sqrtf(p2.w) * 1.01f;
        const float ta = fmaxf(p2.x, -rb), tb = fminf(p2.y, p0.w + rb);
        const float ox = p0.x - F.ox, oy = p0.y - F.oy, oz = p0.z - F.oz;
        const float ax = __builtin_fmaf(p1.x, ta, ox), ay = __builtin_fmaf(p1.y, ta, oy),
                    az = __builtin_fmaf(p1.z, ta, oz);
        const float bx = __builtin_fmaf(p1.x, tb, ox), by = __builtin_fmaf(p1.y, tb, oy),
                    bz = __builtin_fmaf(p1.z, tb, oz);
        // rounding of the endpoints and of the plane distances: 1e-6 of the coordinates involved
        const float em = __builtin_fmaf(
            1e-6f, ((__builtin_fabsf(p0.x) + __builtin_fabsf(p0.y)) + __builtin_fabsf(p0.z)) + (p0.w + rb), F.om);
        // the smallest over the planes of the larger endpoint distance: the segment lies beyond
        // some plane iff it is below -(rb + em)
        float near = INFINITY;
        for (int k = 0; k < 4; ++k) {
            const float* n = F.n[k];
            const float da = __builtin_fmaf(n[2], az, __builtin_fmaf(n[1], ay, n[0] * ax));
            const float db = __builtin_fmaf(n[2], bz, __builtin_fmaf(n[1], by, n[0] * bx));
            near = fminf(near, fmaxf(da, db));
        }
        // end pieces (their ownership range is open) of beams nearly perpendicular to some ray stay
        const float q = __builtin_fmaf(F.mz, p1.z, __builtin_fmaf(F.my, p1.y, F.mx * p1.x));
        const bool end = !(__builtin_isfinite(p2.x) && __builtin_isfinite(p2.y));
        const bool tie = end && !((__builtin_fabsf(q) - F.spread) * rb > 8.0f * em);
        out = near < -(rb + em) && !tie;
    }
    return __ballot((uint32_t)lane < cnt && !out);
}

// The photons [start, start + cnt) of a leaf that some ray of the wave may accept: a photon is
// accepted at a point of a ray with t > min_t >= 0, inside the frustum, within its radius, so a
// photon farther than 1.01 of its radius beyond one of the planes is skipped.
__device__ __forceinline__ uint64_t frustum_photons(const EvalArgs& A, const Frustum& F, uint32_t start,
                                                    uint32_t cnt) {
    const int lane = threadIdx.x & (kWave - 1);
    bool out = false;
    if ((uint32_t)lane < cnt) {
        const float4 p = A.pos_r2[start + lane];
        const float cx = p.x - F.ox, cy = p.y - F.oy, cz = p.z - F.oz;
        // as for beam pieces: hardware square root and fused plane distances, inside the margin
        const float m = __builtin_fmaf(1e-6f, (__builtin_fabsf(p.x) + __builtin_fabsf(p.y)) + __builtin_fabsf(p.z),
                                       __builtin_fmaf(__builtin_amdgcn_sqrtf(p.w), 1.01f, F.om));
        float near = INFINITY;
        for (int k = 0; k < 4; ++k) {
            const float* n = F.n[k];
            near = fminf(near, __builtin_fmaf(n[2], cz, __builtin_fmaf(n[1], cy, n[0] * cx)));
        }
        out = near < -m;
    }
    return __ballot((uint32_t)lane < cnt && !out);
}

template <int MODE>
__device__ __forceinline__ void beam_leaf(const EvalArgs& A, const Ray& r, SegState& s, LaneOut<MODE>& lo,
                                          uint32_t start, uint64_t items, bool short_q) {
    // No software prefetch of the next piece: the rotation of two 64-byte records through
    // SGPRs cost more scalar moves and SGPR pressure than the latency it hid (measured 14 %).
    while (items) {
        const uint32_t i = start + (uint32_t)__builtin_ctzll(items);
        items &= items - 1;
        const PieceDev pc = uniform_at<MODE>(A.pieces, i);
        const uint32_t word = __float_as_uint(pc.p2.z);
        const int32_t bmed = (int32_t)(word & kMediumMask);
        float dist, st, t1, t2, radius;
        // radius = mStartRadius (p1.w) + t2 * mRadiusChange (p3.y)
        const bool hit = test_beam_beam(bmed == s.medium, r.ox, r.oy, r.oz, r.dx, r.dy, r.dz, r.d1o1, s.tmin, s.tmax,
                                        pc.p0.x, pc.p0.y, pc.p0.z, pc.p1.x, pc.p1.y, pc.p1.z, pc.p3.x, pc.p0.w,
                                        pc.p2.w, pc.p2.x, pc.p2.y, pc.p1.w, pc.p3.y, dist, st, t1, t2, radius);
        if ((MODE & 7) == (int)Mode::Upbp) {
            // per-cell reduction: a hit is queued with the times its cell tests it and the
            // cell's pdf, in place of the radius (recomputed from the piece when drained)
            uint32_t red_n = 1;
            float red_pdf = 1.0f;
            if ((MODE & kReduced) && hit)
                red_n = red_decide(A.red, r.qkey, r.ox + r.dx * t1, r.oy + r.dy * t1, r.oz + r.dz * t1, A.orig[i],
                                   red_pdf);
            const bool queue = hit && red_n != 0u;
            const uint64_t m = __ballot(queue);
            if (m) {
                if (queue) {
                    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
                    const uint32_t pos = (lo.qt + lane_rank(m)) & (kHq - 1);
                    lds_write(g_hq[w][0][pos], i);
                    lds_write(g_hq[w][1][pos], (uint32_t)lane | ((word & kShortBeamBit) ? 256u : 0u) | (red_n << 9));
                    lds_write(g_hq[w][2][pos], __float_as_uint(dist));
                    lds_write(g_hq[w][3][pos], __float_as_uint(st));
                    lds_write(g_hq[w][4][pos], __float_as_uint(t1));
                    lds_write(g_hq[w][5][pos], __float_as_uint(t2));
                    lds_write(g_hq[w][6][pos], __float_as_uint((MODE & kReduced) ? red_pdf : radius));
                    lo.hits += red_n;
                }
                lo.qt = uni(lo.qt + (uint32_t)__popcll(m));
                if (lo.qt - lo.qh >= (uint32_t)kWave) drain_beams<MODE>(A, r, s, lo, kWave, short_q);
            }
            continue;
        }
        float red_w = 1.0f;
        uint32_t red_n = 1;
        if ((MODE & kReduced) && hit) {
            // the hit belongs to the reduction grid cell of its query point
            float pdf;
            red_n = red_decide(A.red, r.qkey, r.ox + r.dx * t1, r.oy + r.dy * t1, r.oz + r.dz * t1, A.orig[i], pdf);
            red_w = (1.0f / pdf) * (float)red_n;
        }
        // the adjoint reduces the item gradient over the wave, so every lane enters when one
        // hits; elsewhere the lanes that hit enter on their own (a ballot of this divergent
        // bool would first select it into a VGPR and compare it back)
        const bool take = hit && red_n != 0;
        if ((MODE & 7) == (int)Mode::Adjoint ? __ballot(take) != 0 : take) {
            const float4 flux = uniform_at<MODE>(A.piece_flux, i);
            float gb0 = 0.f, gb1 = 0.f, gb2 = 0.f;
            if (hit && red_n != 0) {
                const bool short_b = (word & kShortBeamBit) != 0;
                const float dq = t1 - s.tmin;
                // T(t1 - tmin) [/ T_k] * T(t2) [/ T_k(t2)], one exponential per channel
                const Trans tr = transmittance(s, dq, t2, short_diff(short_b, short_q));
                const float a0 = tr.c0, a1 = tr.c1, a2 = tr.c2;
                // phase: Evaluate(ray.direction, beam direction), cos = -dot(d2, d1)
                const float ph = lo.aniso ? phase_pdf(s.g, false, -dot3(pc.p1.x, pc.p1.y, pc.p1.z, r.dx, r.dy, r.dz))
                                          : kInvPi * 0.25f;
                // 1D kernel (1 - dist^2/r^2) * 3 / (4 r sin(theta)), PhotonBeam.hxx:364-365
                const float kern = radial_kernel(dist * dist, radius * radius);
                float scale = (ph * kern * 3.0f) * __builtin_amdgcn_rcpf((4.0f * radius) * st);
                if (MODE & kReduced) scale *= red_w;
                const float b0 = a0 * scale, b1 = a1 * scale, b2 = a2 * scale;
                const float c0 = flux.x * s.ss0 * b0, c1 = flux.y * s.ss1 * b1, c2 = flux.z * s.ss2 * b2;
                if ((MODE & 7) == (int)Mode::Adjoint) {
                    gb0 = s.w0 * b0 * s.ss0;
                    gb1 = s.w1 * b1 * s.ss1;
                    gb2 = s.w2 * b2 * s.ss2;
                    s.gs0 += s.w0 * b0 * flux.x;
                    s.gs1 += s.w1 * b1 * flux.y;
                    s.gs2 += s.w2 * b2 * flux.z;
                    const float g0 = s.w0 * c0, g1 = s.w1 * c1, g2 = s.w2 * c2;
                    // log C_c holds -sigma_t_c ((t1 - tmin) + t2) plus, for the SHORT
                    // normalisations by the channel-k transmittance, +sigma_t_k (t1 - tmin)
                    // (SHORT query) and +sigma_t_k t2 (SHORT beam)
                    const float L = dq + t2;
                    s.gt0 -= g0 * L;
                    s.gt1 -= g1 * L;
                    s.gt2 -= g2 * L;
                    const float Lk = (short_q ? dq : 0.f) + (short_b ? t2 : 0.f);
                    if (Lk != 0.f) {
                        const float sum = ((g0 + g1) + g2) * Lk;
                        if (s.kidx == 0) s.gt0 += sum;
                        else if (s.kidx == 1) s.gt1 += sum;
                        else s.gt2 += sum;
                    }
                    s.acc0 += g0;
                    s.acc1 += g1;
                    s.acc2 += g2;
                } else {
                    s.acc0 += c0;
                    s.acc1 += c1;
                    s.acc2 += c2;
                }
                lo.hits++;
                if ((MODE & 7) == (int)Mode::Signature) {
                    lo.sig_n += red_n;
                    lo.sig_h += red_n * hash32(A.orig[i]);
                }
            }
            if ((MODE & 7) == (int)Mode::Adjoint) add_item_gradient(A.grad_items, A.orig[i], gb0, gb1, gb2);
        }
    }
}

// ---- pair queue of waves without a common origin -----------------------------
// The rays of scattered paths share a wave but no direction: of 64 lanes only one or two meet the box of
// a visited leaf (200k rays from points of the media: 47 million pieces with a ray within the radius
// of their line, 1.9 rays each), so testing an item with the whole wave leaves nearly all lanes idle.
// Where at most kSparseLanes lanes meet a leaf's box, its (lane, item) pairs are queued instead and
// tested 64 at a time, a lane taking any ray and any item. An item is accepted only by rays that meet
// its box (the boxes are widened for that), but for the pairs that a beam's first and last piece own
// beyond its ends: those pieces are tested by the whole wave as ever.
// Photons gain even in the smallest structures; beams of fewer than kSparseFrom pieces don't make up for
// the second launch (6000 parallel rays x 200 beams 90 us in one launch, 97 in two; 700 and 6000 scattered
// rays the same either way).
constexpr int kSparseLanes = 16;
constexpr int64_t kSparseFrom = 1024;
constexpr int kPq = 128;  // a leaf adds at most 64 pairs per lane to fewer than 64 queued
__shared__ uint32_t g_pq[kHqWaves][2][kPq];

// Tests the first n (1..64) queued pairs: [0] item, [1] lane.
template <int EST, int MODE>
__device__ __forceinline__ void drain_pairs(const EvalArgs& A, const Ray& r, const SegState& s, LaneOut<MODE>& lo,
                                            uint32_t n, bool short_q) {
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const uint32_t pos = (lo.qh + (uint32_t)lane) & (kPq - 1);
    const bool act = (uint32_t)lane < n;
    const int owner = act ? (int)(lds_read(g_pq[w][1][pos]) & (kWave - 1)) : lane;
    const uint32_t i = lds_read(g_pq[w][0][pos]);
    const float ox = from_lane(r.ox, owner), oy = from_lane(r.oy, owner), oz = from_lane(r.oz, owner);
    const float dx = from_lane(r.dx, owner), dy = from_lane(r.dy, owner), dz = from_lane(r.dz, owner);
    const float tmin = from_lane(s.tmin, owner), tmax = from_lane(s.tmax, owner);
    SegState so;
    so.x0 = from_lane(s.x0, owner);
    so.x1 = from_lane(s.x1, owner);
    so.x2 = from_lane(s.x2, owner);
    so.ek = from_lane(s.ek, owner);
    const float ss0 = from_lane(s.ss0, owner), ss1 = from_lane(s.ss1, owner), ss2 = from_lane(s.ss2, owner);
    const float g = from_lane(s.g, owner);
    bool hit;
    float c0 = 0.f, c1 = 0.f, c2 = 0.f;
    if (EST == kEstPhotons) {
        float t, sq;
        const float4 p = A.pos_r2[act ? i : 0u];
        hit = act && test_bre(ox, oy, oz, dx, dy, dz, tmin, tmax, p.x, p.y, p.z, p.w, t, sq);
        if (hit && (MODE & 7) == (int)Mode::Forward) {
            const float4 pw = A.power[i];
            const float dt = t - tmin;
            const Trans tr = transmittance(so, dt);
            float ph = kInvPi * 0.25f;
            if (lo.aniso) {
                const float4 in = A.inc[i];
                ph = phase_pdf(g, false, dot3(in.x, in.y, in.z, dx, dy, dz));
            }
            const float scale = (ph * radial_kernel(sq, p.w)) * pw.w;
            c0 = pw.x * (tr.c0 * scale) * ss0;
            c1 = pw.y * (tr.c1 * scale) * ss1;
            c2 = pw.z * (tr.c2 * scale) * ss2;
        }
    } else {
        const float d1o1 = from_lane(r.d1o1, owner);
        const int32_t medium = from_lane(s.medium, owner);
        const PieceDev pc = A.pieces[act ? i : 0u];
        const uint32_t word = __float_as_uint(pc.p2.z);
        float dist, st, t1, t2, radius;
        hit = test_beam_beam(act && (int32_t)(word & kMediumMask) == medium, ox, oy, oz, dx, dy, dz, d1o1, tmin, tmax,
                             pc.p0.x, pc.p0.y, pc.p0.z, pc.p1.x, pc.p1.y, pc.p1.z, pc.p3.x, pc.p0.w, pc.p2.w, pc.p2.x,
                             pc.p2.y, pc.p1.w, pc.p3.y, dist, st, t1, t2, radius);
        if (hit && (MODE & 7) == (int)Mode::Forward) {
            const float4 flux = A.piece_flux[i];
            const float dq = t1 - tmin;
            const Trans tr = transmittance(so, dq, t2, short_diff((word & kShortBeamBit) != 0, short_q));
            const float ph = lo.aniso ? phase_pdf(g, false, -dot3(pc.p1.x, pc.p1.y, pc.p1.z, dx, dy, dz))
                                      : kInvPi * 0.25f;
            const float kern = radial_kernel(dist * dist, radius * radius);
            const float scale = (ph * kern * 3.0f) * __builtin_amdgcn_rcpf((4.0f * radius) * st);
            c0 = flux.x * ss0 * (tr.c0 * scale);
            c1 = flux.y * ss1 * (tr.c1 * scale);
            c2 = flux.z * ss2 * (tr.c2 * scale);
        }
    }
    if (hit) {
        lo.hits++;
        if ((MODE & 7) == (int)Mode::Signature) {
            uint32_t* sums = reinterpret_cast<uint32_t*>(&g_hacc[w][0][0]);
            atomicAdd(&sums[owner], 1u);
            atomicAdd(&sums[kWave + owner], hash32(A.orig[i]));
        } else {
            atomicAdd(&g_hacc[w][0][owner], c0);
            atomicAdd(&g_hacc[w][1][owner], c1);
            atomicAdd(&g_hacc[w][2][owner], c2);
        }
    }
    lo.qh += n;
}

// Queues the pairs of the lanes of `lanes` with the items start + j, j the bits of items.
template <int EST, int MODE>
__device__ __forceinline__ void queue_pairs(const EvalArgs& A, const Ray& r, const SegState& s, LaneOut<MODE>& lo,
                                            uint64_t lanes, uint32_t start, uint64_t items, bool short_q) {
    if (!items) return;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const uint32_t n = (uint32_t)__popcll(items), rank = lane_rank(items);
    while (lanes) {
        const uint32_t owner = (uint32_t)__builtin_ctzll(lanes);
        lanes &= lanes - 1;
        if ((items >> lane) & 1u) {
            const uint32_t pos = (lo.qt + rank) & (kPq - 1);
            lds_write(g_pq[w][0][pos], start + (uint32_t)lane);
            lds_write(g_pq[w][1][pos], owner);
        }
        lo.qt = uni(lo.qt + n);
        if (lo.qt - lo.qh >= (uint32_t)kWave) drain_pairs<EST, MODE>(A, r, s, lo, kWave, short_q);
    }
}

// End of a segment: tests what is still queued and moves the owners' sums to their lanes.
template <int EST, int MODE>
__device__ __forceinline__ void sparse_segment_end(const EvalArgs& A, const Ray& r, SegState& s, LaneOut<MODE>& lo,
                                                   bool short_q) {
    const uint32_t n = uni(lo.qt - lo.qh);
    if (n) drain_pairs<EST, MODE>(A, r, s, lo, n, short_q);
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    if ((MODE & 7) == (int)Mode::Signature) {
        lo.sig_n += __float_as_uint(lds_read(g_hacc[w][0][lane]));
        lo.sig_h += __float_as_uint(lds_read(g_hacc[w][1][lane]));
    } else {
        s.acc0 += lds_read(g_hacc[w][0][lane]);
        s.acc1 += lds_read(g_hacc[w][1][lane]);
        s.acc2 += lds_read(g_hacc[w][2][lane]);
    }
    for (int c = 0; c < 3; ++c) lds_write(g_hacc[w][c][lane], 0.f);
}

// Bits j of the pieces start + j (j < 64) that are a beam's first or last.
__device__ __forceinline__ uint64_t end_pieces(const EvalArgs& A, uint32_t start) {
    const uint64_t lo = A.end_bits[start >> 6], hi = A.end_bits[(start >> 6) + 1u];
    const uint32_t sh = start & 63u;
    return sh ? (lo >> sh) | (hi << (64u - sh)) : lo;
}

// ---- wave-cooperative traversal ------------------------------------------
// The items [start, start + cnt) (cnt <= 64) of a leaf that the rays of `lanes` meet the box of, culled
// against the wave's frustum first when it has one. tested: the items that the whole wave tests.
template <int EST, int MODE>
__device__ __forceinline__ void visit_leaf(const EvalArgs& A, const Frustum& F, bool fr, ItemPart part,
                                           uint64_t lanes, const Ray& r, SegState& s, LaneOut<MODE>& lo,
                                           uint32_t start, uint32_t cnt, bool short_q, uint32_t& tested) {
    const uint64_t all = (MODE & kSplit) ? part.items(start, cnt) : cnt >= 64u ? ~0ull : ((1ull << cnt) - 1ull);
    if ((MODE & kSparse) && __popcll(lanes) <= kSparseLanes) {
        const uint64_t ends = EST == kEstPhotons ? 0ull : end_pieces(A, start) & all;
        tested += (uint32_t)__popcll(ends);
        if (EST == kEstBeams) beam_leaf<MODE>(A, r, s, lo, start, ends, short_q);
        queue_pairs<EST, MODE>(A, r, s, lo, lanes, start, all & ~ends, short_q);
    } else if (EST == kEstPhotons) {
        const uint64_t items = fr ? frustum_photons(A, F, start, cnt) & all : all;
        tested += (uint32_t)__popcll(items);
        photon_leaf<MODE>(A, r, s, lo, start, items, short_q);
    } else {
        const uint64_t items = fr ? frustum_items(A, F, start, cnt) & all : all;
        tested += (uint32_t)__popcll(items);
        beam_leaf<MODE>(A, r, s, lo, start, items, short_q);
    }
}

template <int EST, int MODE>
__device__ __forceinline__ void traverse(const EvalArgs& A, ItemPart part, const Ray& r, SegState& s,
                                         LaneOut<MODE>& lo, bool short_q, uint32_t& nodes_visited, uint64_t& tests,
                                         uint32_t& overflow) {
    const int lane = threadIdx.x & (kWave - 1);
    uint32_t stk0 = 0, stk1 = 0;
    int sp = 0;
    uint32_t node = A.root;
    uint32_t tested = 0;
    const uint32_t queued = lo.qt;
    Frustum F;
    const bool fr = !(MODE & kSparse) && make_frustum(r, s, F);
    while (true) {
        node = uni(node);
        // One 64-byte scalar load for the whole node, then both slab tests without
        // short-circuit: testing the child references first would make the box loads
        // wait on them (three dependent scalar round trips per node instead of one).
        const NodeDev nd = uniform_at<MODE>(A.nodes, node);
        const float4 a = nd.a, b = nd.b, c = nd.c;
        const uint4 rr = nd.r;
        nodes_visited++;
        const uint64_t m0 = slab_mask(r, s.tmin, s.tmax, a.x, a.y, a.z, a.w, b.x, b.y);
        const uint64_t m1 = slab_mask(r, s.tmin, s.tmax, b.z, b.w, c.x, c.y, c.z, c.w);
        // the wave-uniform child references and the items their subtrees hold (this wave's part
        // or not) are tested on the scalar side
        const uint32_t n0 = rr.z & kSpanMask, n1 = rr.w & kSpanMask;
        const uint32_t s0 = (rr.z & kSpanEnds) ? rr.x + 1u - n0 : rr.x;
        const uint32_t s1 = (rr.w & kSpanEnds) ? rr.y + 1u - n1 : rr.y;
        const bool any0 = m0 != 0 && rr.z != kInvalid && (!(MODE & kSplit) || part.meets(s0, n0));
        const bool any1 = m1 != 0 && rr.w != kInvalid && (!(MODE & kSplit) || part.meets(s1, n1));
        // A leaf; or, for a wave with a frustum, an inner node whose subtree holds at most
        // frustum_leaf items: the frustum check takes a whole leaf in one pass, so a small
        // subtree costs less as one leaf than as nodes (leaves stay small for the other waves).
        const bool leaf0 = any0 && (!(rr.z & kInner) || (fr && n0 <= A.frustum_leaf));
        const bool leaf1 = any1 && (!(rr.w & kInner) || (fr && n1 <= A.frustum_leaf));
        if (leaf0) visit_leaf<EST, MODE>(A, F, fr, part, m0, r, s, lo, s0, n0, short_q, tested);
        if (leaf1) visit_leaf<EST, MODE>(A, F, fr, part, m1, r, s, lo, s1, n1, short_q, tested);
        const bool go0 = any0 && !leaf0;
        const bool go1 = any1 && !leaf1;
        if (go0 && go1) {
            if (sp >= kStackMax) {
                overflow++;
                break;
            }
            if (sp < kWave)
                stk0 = (lane == sp) ? rr.y : stk0;
            else
                stk1 = (lane == sp - kWave) ? rr.y : stk1;
            ++sp;
            node = rr.x;
        } else if (go0) {
            node = rr.x;
        } else if (go1) {
            node = rr.y;
        } else {
            if (sp == 0) break;
            --sp;
            node = sp < kWave ? (uint32_t)__builtin_amdgcn_readlane((int)stk0, sp)
                              : (uint32_t)__builtin_amdgcn_readlane((int)stk1, sp - kWave);
        }
    }
    tests += (uint64_t)tested * (uint32_t)__popcll(__ballot(s.tmin <= s.tmax));
    if (MODE & kSparse) tests += lo.qt - queued;  // pairs
}

__device__ __forceinline__ bool finite3(float x, float y, float z) {
    return __builtin_isfinite(x) && __builtin_isfinite(y) && __builtin_isfinite(z);
}

// The block's row of the medium gradients (media_base is 0 outside batched plans, which have no adjoint).
__device__ __forceinline__ float* grad_row(const EvalArgs& A) {
    return as_global(A.grad_media) + (size_t)(blockIdx.x & A.grad_mask) * A.n_media * 6;
}

// A lane's query: whether its ray is evaluated (its offsets are in order and its numbers finite), else
// with the error bits that say why not. Zeros for a lane past the last query.
struct QueryIn {
    float o[3], d[3];
    int64_t s0;
    int nseg;
    uint32_t qi, err;  // fewer than 2^32 queries
    bool alive;
};
__device__ __forceinline__ QueryIn read_query(const EvalArgs& A, int64_t slot) {
    QueryIn q = {};
    if (slot >= A.count) return q;
    q.qi = A.perm ? A.perm[slot] : (uint32_t)slot;
    const float* o = A.origin + 3 * (int64_t)q.qi;
    const float* d = A.direction + 3 * (int64_t)q.qi;
    for (int a = 0; a < 3; ++a) {
        q.o[a] = o[a];
        q.d[a] = d[a];
    }
    q.s0 = A.offsets[q.qi];
    const int64_t s1 = A.offsets[(int64_t)q.qi + 1], sq = A.offsets[A.count];
    q.nseg = (int)(s1 - q.s0);
    q.alive = true;
    if (!(q.s0 >= 0 && q.s0 <= s1 && s1 <= sq)) {
        q.err |= kErrBadOffsets;
        q.alive = false;
    }
    if (!finite3(q.o[0], q.o[1], q.o[2]) || !finite3(q.d[0], q.d[1], q.d[2])) {
        q.err |= kErrNonFinite;
        q.alive = false;
    }
    return q;
}

// Whether the rays of the lanes with `on` start at the point of their first (true of none).
__device__ __forceinline__ uint64_t start_elsewhere(const QueryIn& q, bool on, int first) {
    const float ox = __shfl(q.o[0], first, kWave), oy = __shfl(q.o[1], first, kWave), oz = __shfl(q.o[2], first, kWave);
    return __ballot(on && !(q.o[0] == ox && q.o[1] == oy && q.o[2] == oz));
}

// Whether a ray has a segment of a scattering medium (the walk ends at a bad medium, as the gather does).
__device__ __forceinline__ bool gathers(const EvalArgs& A, const QueryIn& q) {
    for (int k = 0; k < q.nseg; ++k) {
        const int32_t m = A.segments[q.s0 + k].medium_id;
        if (m < 0 || m >= A.n_media) return false;
        if (A.media[A.media_base + m].has_scattering) return true;
    }
    return false;
}

// Whether those of the wave's rays that gather anything start at one point (true of none): rays that miss
// the media or have ended may start anywhere (a frame padded with them keeps its frusta). This one answer
// says which of the two launches (in_two) a tile belongs to: the launches themselves and the tile plan,
// which gives tasks and rows to the tiles of the first, all take it from here. No segment is read where all
// evaluated rays start at one point, and those of two rays where these show that the answer is no: reading
// all 64 cost the launches of rays without a common origin up to 10 % (1M parallel rays x 50k photons 666
// -> 736 us).
__device__ __forceinline__ bool common_origin(const EvalArgs& A, const QueryIn& q) {
    const uint64_t am = __ballot(q.alive);
    const int first = am ? __builtin_ctzll(am) : 0;
    const uint64_t apart = start_elsewhere(q, q.alive, first);
    if (!apart) return true;
    uint64_t look = (1ull << first) | (apart & (0ull - apart)), on = 0;
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass, look = am) {
        const bool mine = (look >> (threadIdx.x & (kWave - 1))) & 1u;
        on = __ballot(mine && gathers(A, q));
        if (pass == 0 && on == look) return false;
    }
    return start_elsewhere(q, (on >> (threadIdx.x & (kWave - 1))) & 1u, on ? __builtin_ctzll(on) : 0) == 0;
}

__shared__ float g_part[4][3][kWave];  // the sums of a split launch's waves

// Processes the 64 queries of one tile (wave) against its part of the items. `slot0` is the first
// lane slot. False: the tile is the other launch's (in_two), nothing was done.
template <int EST, int MODE, bool KARG>
__device__ bool run_tile(const EvalArgs& A, int64_t slot0, ItemPart part, unsigned long long* local_stats,
                         float* lds_media /* adjoint: [lds_media_n][6][64] for this wave or null */) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t slot = slot0 + lane;
    const bool valid = slot < A.count;
    const QueryIn in = read_query(A, slot);
    const uint32_t qi = in.qi;
    uint32_t err = in.err;
    Ray r = {};
    r.ox = in.o[0], r.oy = in.o[1], r.oz = in.o[2];
    r.dx = in.d[0], r.dy = in.d[1], r.dz = in.d[2];
    int nseg = in.nseg;
    bool alive = in.alive;
    if (KARG && in_two(MODE) && !A.known && common_origin(A, in) == ((MODE & kSparse) != 0)) return false;
    r.ix = guard_inv(r.dx);
    r.iy = guard_inv(r.dy);
    r.iz = guard_inv(r.dz);
    r.oix = r.ox * r.ix;
    r.oiy = r.oy * r.iy;
    r.oiz = r.oz * r.iz;
    r.d1o1 = dot3(r.dx, r.dy, r.dz, r.ox, r.oy, r.oz);
    if (MODE & kReduced) {
        const uint32_t bits[6] = {__float_as_uint(r.ox), __float_as_uint(r.oy), __float_as_uint(r.oz),
                                  __float_as_uint(r.dx), __float_as_uint(r.dy), __float_as_uint(r.dz)};
        r.qkey = red_query_key(bits);
    }
    if (!alive) nseg = 0;
    int maxseg = nseg;
    for (int off = 32; off > 0; off >>= 1) maxseg = max(maxseg, __shfl_xor(maxseg, off, kWave));
    maxseg = (int)uni((uint32_t)maxseg);

    const bool short_q = A.short_query != 0;
    float P0 = 1.f, P1 = 1.f, P2 = 1.f;
    float R0 = 0.f, R1 = 0.f, R2 = 0.f;
    float W0 = 0.f, W1 = 0.f, W2 = 0.f;
    if ((MODE & 7) == (int)Mode::Adjoint && valid) {
        W0 = A.grad_out[3 * (int64_t)qi];
        W1 = A.grad_out[3 * (int64_t)qi + 1];
        W2 = A.grad_out[3 * (int64_t)qi + 2];
    }
    LaneOut<MODE> lo;
    if ((MODE & 7) == (int)Mode::Upbp) {
        // per-query AdditionalRayDataForMis (Bre.cxx:842-849 runs it per segment below)
        lo.ml.tail = CamTail{0.f, 0.f, 0u};
        lo.ml.cam_len = 1;
        lo.ml.ray_flags = 0;
        lo.ml.last_pdf_w_inv = 1.f;
        lo.ml.pref_pdf = 1.f;
        lo.ml.pref_rev = 1.f;
        lo.ml.seg_flags = UPBP_END_IN_MEDIUM;
        if (valid) {
            const upbp_query_mis qm = A.qmis[qi];
            if (qm.camera_path_length < 1 || qm.camera_offset < 0 ||
                qm.camera_offset + (int64_t)qm.camera_path_length >= A.mis.camera_count) {
                err |= kBadLightIndex;
                alive = false;
                nseg = 0;
            } else {
                lo.ml.cam_len = (int)qm.camera_path_length;
                lo.ml.tail = camera_tail(A.mis.camera + qm.camera_offset, lo.ml.cam_len, A.mis.p.query_beam_type,
                                         A.mis.p.photon_beam_type, A.mis.p.techniques);
                lo.ml.ray_flags = qm.ray_sampling_flags;
                lo.ml.last_pdf_w_inv = qm.last_pdf_w_inv;
            }
        }
    }
    if ((MODE & 7) == (int)Mode::Upbp || (MODE & kSparse)) {
        const int w = threadIdx.x / kWave;
        lds_write(g_hacc[w][0][lane], 0.f);
        lds_write(g_hacc[w][1][lane], 0.f);
        lds_write(g_hacc[w][2][lane], 0.f);
    }
    uint64_t tests = 0;
    uint32_t nodes_visited = 0, overflow = 0;
    for (int k = 0; k < maxseg; ++k) {
        bool has = alive && k < nseg;
        SegState s;
        s.tmin = __builtin_inff();
        s.tmax = -__builtin_inff();
        s.x0 = s.x1 = s.x2 = s.ek = 0.f;
        s.ss0 = s.ss1 = s.ss2 = 0.f;
        s.g = 0.f;
        s.kidx = 0;
        s.medium = -1;
        s.acc0 = s.acc1 = s.acc2 = 0.f;
        s.w0 = s.w1 = s.w2 = 0.f;
        s.gs0 = s.gs1 = s.gs2 = 0.f;
        s.gt0 = s.gt1 = s.gt2 = 0.f;
        const EvalArgs& C = *reread<KARG>(A, (uint32_t)k);
        const upbp_volume_segment* segments = as_global(C.segments);
        const MediumDev* media = as_global(C.media);
        bool scatter = false;
        if (has) {
            const upbp_volume_segment* sg = segments + (as_global(C.offsets)[qi] + k);
            const float tmin = sg->dist_min, tmax = sg->dist_max;
            const int32_t mid = sg->medium_id;
            const float a0 = sg->attenuation[0], a1 = sg->attenuation[1], a2 = sg->attenuation[2];
            const float pdf = sg->ray_sample_pdf;
            // n_media counts the media from media_base on (the whole table outside batched plans)
            if (mid < 0 || mid >= C.n_media) {
                err |= kErrBadMedium;
                has = false;
                alive = false;
            } else if (!__builtin_isfinite(tmin) || !__builtin_isfinite(tmax) || !finite3(a0, a1, a2) ||
                       !__builtin_isfinite(pdf)) {
                err |= kErrNonFinite;
                has = false;
                alive = false;
            } else if (tmin > tmax) {
                err |= kErrBadSegment;
                has = false;
                alive = false;
            } else {
                const MediumDev* m = media + (C.media_base + mid);
                scatter = m->has_scattering != 0;
                s.medium = mid;
                if (scatter) {
                    s.tmin = tmin;
                    s.tmax = tmax;
                    set_factors(s, m->st[0], m->st[1], m->st[2], m->min_idx, short_q);
                    s.ss0 = m->ss[0];
                    s.ss1 = m->ss[1];
                    s.ss2 = m->ss[2];
                    s.g = m->isotropic ? 0.f : m->g;
                    s.kidx = m->min_idx;
                    s.min_comp = m->min_comp;
                    s.mfp = m->mfp;
                    s.cont = m->cont;
                }
                if ((MODE & 7) == (int)Mode::Upbp)
                    lo.ml.seg_flags = UPBP_END_IN_MEDIUM | (k == 0 ? lo.ml.ray_flags : 0u);
            }
        }
        if ((MODE & 7) == (int)Mode::Adjoint) {
            s.w0 = W0 * P0;
            s.w1 = W1 * P1;
            s.w2 = W2 * P2;
        }
        if (__ballot(scatter)) {
            lo.aniso = __ballot(s.g != 0.f) != 0;
            traverse<EST, MODE>(A, part, r, s, lo, short_q, nodes_visited, tests, overflow);
            if ((MODE & 7) == (int)Mode::Upbp) upbp_segment_end<EST, MODE>(A, r, s, lo, short_q);
            if (MODE & kSparse) sparse_segment_end<EST, MODE>(A, r, s, lo, short_q);
        }
        const EvalArgs& D = *reread<KARG>(A, nodes_visited);
        if (has) {
            R0 += P0 * s.acc0;
            R1 += P1 * s.acc1;
            R2 += P2 * s.acc2;
            if ((MODE & 7) == (int)Mode::Adjoint && scatter) {
                // medium gradients of this segment plus the prefix terms of earlier segments
                const int mloc = D.media_base + s.medium;
                float* slab_m = (lds_media && s.medium < D.lds_media_n) ? lds_media : nullptr;
                if (slab_m) {
                    float* base = slab_m + (size_t)s.medium * 6 * kWave + lane;
                    base[0 * kWave] += s.gs0;
                    base[1 * kWave] += s.gs1;
                    base[2 * kWave] += s.gs2;
                    base[3 * kWave] += s.gt0;
                    base[4 * kWave] += s.gt1;
                    base[5 * kWave] += s.gt2;
                } else {
                    float* gm = grad_row(D) + (size_t)mloc * 6;
                    unsafeAtomicAdd(&gm[0], s.gs0);
                    unsafeAtomicAdd(&gm[1], s.gs1);
                    unsafeAtomicAdd(&gm[2], s.gs2);
                    unsafeAtomicAdd(&gm[3], s.gt0);
                    unsafeAtomicAdd(&gm[4], s.gt1);
                    unsafeAtomicAdd(&gm[5], s.gt2);
                }
                // s.acc = sum_hits w * C for this segment (w already includes P)
                for (int j = 0; j < k; ++j) {
                    const upbp_volume_segment* sp = as_global(D.segments) + (as_global(D.offsets)[qi] + j);
                    const float len = sp->dist_max - sp->dist_min;
                    const int32_t mj = sp->medium_id;
                    float d0 = -s.acc0 * len, d1 = -s.acc1 * len, d2 = -s.acc2 * len;
                    // SHORT query: the segment's factor is attenuation over its pass-through pdf
                    // exp(-sigma_t_k len) when the medium samples distances (Media.hxx:294-323)
                    if (short_q && !D.lite) {
                        const MediumDev* mm = as_global(D.media) + (D.media_base + mj);
                        if (mm->min_comp > 0.f && mm->has_scattering) {
                            const float sum = ((s.acc0 + s.acc1) + s.acc2) * len;
                            if (mm->min_idx == 0) d0 += sum;
                            else if (mm->min_idx == 1) d1 += sum;
                            else d2 += sum;
                        }
                    }
                    if (lds_media && mj < D.lds_media_n) {
                        float* base = lds_media + (size_t)mj * 6 * kWave + lane;
                        base[3 * kWave] += d0;
                        base[4 * kWave] += d1;
                        base[5 * kWave] += d2;
                    } else {
                        float* gm = grad_row(D) + (size_t)(D.media_base + mj) * 6;
                        unsafeAtomicAdd(&gm[3], d0);
                        unsafeAtomicAdd(&gm[4], d1);
                        unsafeAtomicAdd(&gm[5], d2);
                    }
                }
            }
            // the segment's record is read again here instead of held through the traversal
            const upbp_volume_segment* sg = as_global(D.segments) + (as_global(D.offsets)[qi] + k);
            const MediumDev* m = as_global(D.media) + (D.media_base + s.medium);
            float a0 = sg->attenuation[0], a1 = sg->attenuation[1], a2 = sg->attenuation[2];
            const float pdf = sg->ray_sample_pdf;
            if (D.lite) {
                const float len = sg->dist_max - sg->dist_min;
                a0 = fast_exp(-m->st[0] * len);
                a1 = fast_exp(-m->st[1] * len);
                a2 = fast_exp(-m->st[2] * len);
            }
            if (D.lite || !short_q) {
                P0 *= a0;
                P1 *= a1;
                P2 *= a2;
            } else {
                P0 *= a0 / pdf;
                P1 *= a1 / pdf;
                P2 *= a2 / pdf;
            }
            if (!(P0 > 1e-20f && P1 > 1e-20f && P2 > 1e-20f)) alive = false;
            if ((MODE & 7) == (int)Mode::Upbp) {
                // ray-sampling pdf prefixes of the segment loop (Bre.cxx:871-873, lite :955-958)
                if (D.lite) {
                    float rev = 1.f, spdf = 1.f;
                    if (m->min_comp != 0.f && m->has_scattering) {
                        float att = fmaxf(__expf(-m->min_comp * (sg->dist_max - sg->dist_min)), 1e-35f);
                        const float minatt = m->min_comp * att;
                        const uint32_t f = k == 0 ? lo.ml.ray_flags : 0u;
                        spdf = (f & UPBP_END_IN_MEDIUM) ? minatt : att;
                        rev = (f & UPBP_ORIGIN_IN_MEDIUM) ? minatt : att;
                    }
                    lo.ml.pref_pdf *= spdf;
                    lo.ml.pref_rev *= rev;
                } else {
                    lo.ml.pref_pdf *= pdf;
                    lo.ml.pref_rev *= sg->ray_sample_rev_pdf;
                }
            }
        }
    }
    err |= lo.err;
    const EvalArgs& E = *reread<KARG>(A, nodes_visited);
    if (valid && (MODE & 7) != (int)Mode::Adjoint) {
        if (MODE & kSplit) {  // k_eval stores them
            const int w = threadIdx.x / kWave;
            if ((MODE & 7) == (int)Mode::Signature) {
                g_part[w][0][lane] = __uint_as_float(lo.sig_n);
                g_part[w][1][lane] = __uint_as_float(lo.sig_h);
            } else {
                g_part[w][0][lane] = R0;
                g_part[w][1][lane] = R1;
                g_part[w][2][lane] = R2;
            }
        } else if ((MODE & 7) == (int)Mode::Signature) {
            uint32_t* sig = as_global(E.sig);
            sig[2 * (int64_t)qi] = lo.sig_n;
            sig[2 * (int64_t)qi + 1] = lo.sig_h;
        } else {
            float* out = as_global(E.out) + 3 * (int64_t)qi;
            out[0] = R0;
            out[1] = R1;
            out[2] = R2;
        }
    }
    // per-wave counters
    // Reduced over the wave and made scalar: the running counters then live in SGPRs,
    // not in 64-bit VGPR pairs held across every tile of a persistent wave.
    uint32_t h = lo.hits;
    for (int off = 32; off > 0; off >>= 1) h += __shfl_xor(h, off, kWave);
    uint32_t e = err;
    for (int off = 32; off > 0; off >>= 1) e |= __shfl_xor(e, off, kWave);
    local_stats[EST == kEstPhotons ? kStatPhotonHits : kStatBeamHits] += uni(h);
    local_stats[EST == kEstPhotons ? kStatPhotonCands : kStatBeamCands] += uni_u64(tests);
    local_stats[kStatNodes] += uni(nodes_visited);
    local_stats[kStatError] |= uni(e);
    local_stats[kStatOverflow] += uni(overflow);
    return true;
}

// One wave's counters, in a row of its block's.
__device__ __forceinline__ void flush_stats(const EvalArgs& A, const unsigned long long* ls) {
    if ((threadIdx.x & (kWave - 1)) == 0) {
        unsigned long long* stats = as_global(A.stats) + blockIdx.x % kStatRows * kStatSlots;
        for (int k = 0; k < kStatSlots; ++k) {
            if (k == kStatError) {
                if (ls[k]) atomicOr(&stats[k], ls[k]);
            } else if (ls[k]) {
                atomicAdd(&stats[k], ls[k]);
            }
        }
    }
}

// XCD-aware block order: the hardware deals consecutive workgroups round-robin
// over 8 XCDs; remap so that each XCD works on one contiguous range of tiles
// (neighbouring tiles share nodes and leaves in that XCD's L2).
__device__ __forceinline__ int64_t xcd_block(int64_t bid, int64_t nblk) {
    const int64_t q = nblk / 8, rmd = nblk % 8;
    const int64_t xcd = bid % 8, local = bid / 8;
    return xcd < rmd ? xcd * (q + 1) + local : rmd * (q + 1) + (xcd - rmd) * q + local;
}

// The same in rounds of 8 * chunk blocks: each XCD gets chunk consecutive blocks of every round. Tiles
// cost very unequal times and neighbours cost alike, so one range per XCD left half of the XCDs idle for
// the last third of a launch; 16 neighbouring tiles at a time still share an L2. Beams and photons of
// 1920x1080 rays: 10.9 ms with one range per XCD, 9.04 / 9.00 / 8.95 / 8.87 ms with chunks of 1 / 4 / 16 /
// 64 blocks; a million rays on two million beams: 55.4, 46.0 / 45.5 / 47.1 / 49.0 ms.
constexpr int64_t kXcdChunk = 4;  // blocks of 4 waves; as many tiles of smaller blocks
__device__ __forceinline__ int64_t xcd_round_block(int64_t bid, int64_t nblk, int64_t chunk) {
    const int64_t first = bid / (8 * chunk) * (8 * chunk);
    const int64_t left = nblk - first;
    return first + xcd_block(bid - first, left < 8 * chunk ? left : 8 * chunk);
}

// Forward kernels ask for 8 resident waves per SIMD (64 VGPRs): a few bytes of
// register spill cost less than the latency the extra wave hides (measured 3-4 %).
// UPBP kernels ask for 4 (128 VGPRs), which both fit without spilling.
template <int EST, int MODE>
__global__ __launch_bounds__(256, ((MODE & 7) == (int)Mode::Upbp ? 4 : (MODE & 7) == (int)Mode::Adjoint ? 1 : (MODE & kReduced) ? 6 : (MODE & kSparse) ? 5 : (MODE & 7) == (int)Mode::Forward ? 8 : 1)) void k_eval(
    EvalArgs A) {
    const int wave_in_block = threadIdx.x / kWave;
    const int waves_per_block = blockDim.x / kWave;
    // the parts of a split without a plan are spread over the blocks already
    const int64_t blk = (MODE & kSplit) && !A.tasks ? xcd_block(blockIdx.x, gridDim.x)
                                                    : xcd_round_block(blockIdx.x, gridDim.x, kXcdChunk * 4 / waves_per_block);
    // wave-uniform (fewer than 2^32 waves: at most 2^26 tiles, and splits only of small batches)
    const uint32_t w = uni((uint32_t)(blk * waves_per_block + wave_in_block));
    if ((MODE & kSplit) && A.tasks && w >= as_global(A.plan)->n_tasks) return;
    unsigned long long ls[kStatSlots] = {0, 0, 0, 0, 0, 0, 0, 0};
    // adjoint: per-lane medium gradient slabs, [lds_media_n][6][64] floats per wave, sized at launch
    extern __shared__ float lds_dyn[];
    float* my_lds = nullptr;
    if ((MODE & 7) == (int)Mode::Adjoint) {
        const int slab = A.lds_media_n * 6 * kWave;
        my_lds = lds_dyn + (size_t)wave_in_block * slab;
        for (int k = threadIdx.x & (kWave - 1); k < slab; k += kWave) my_lds[k] = 0.f;
    }
    ItemPart part = {0u, 0u, 6u};
    uint32_t tile = w;
    if (MODE & kSplit) {
        const TileTask t = tile_task(as_global(A.tasks), A.log_parts, A.row0, A.shift, w);
        tile = t.tile;
        part = t.part;
    }
    const int64_t slot0 = (int64_t)tile * kWave;
    if ((MODE & kSparse) && A.tile_class && (slot0 >= A.count || as_global(A.tile_class)[tile] != kCostOther)) return;
    const bool ran = slot0 < A.count && run_tile<EST, MODE, true>(A, slot0, part, ls, my_lds);
    if (in_two(MODE) && !ran) return;
    const EvalArgs& E = *reread<true>(A, (uint32_t)ls[kStatNodes]);
    if ((MODE & 7) != (int)Mode::Adjoint && (MODE & kSplit)) {
        constexpr int kN = (MODE & 7) == (int)Mode::Signature ? 2 : 3;
        const TileTask t = tile_task(as_global(E.tasks), E.log_parts, E.row0, E.shift, w);
        const int lane = threadIdx.x & (kWave - 1);
        const int64_t slot = (int64_t)t.tile * kWave + lane;
        if (slot < E.count) {
            float* out;
            int64_t step = 1;
            if (t.log_parts == 0) {
                out = (kN == 2 ? (float*)as_global(E.sig) : as_global(E.out)) +
                      kN * (E.perm ? (int64_t)as_global(E.perm)[slot] : slot);
            } else {
                out = as_global(E.rows) + (size_t)t.row * kN * kWave + lane;
                step = kWave;
            }
            for (int c = 0; c < kN; ++c) out[c * step] = g_part[wave_in_block][c][lane];
        }
    }
    if ((MODE & 7) == (int)Mode::Adjoint) {
        // reduce the per-lane medium slabs of this wave and add them once
        const int lane = threadIdx.x & (kWave - 1);
        const int nm = E.lds_media_n;
        for (int e = 0; e < nm * 6; ++e) {
            const float v = wave_sum_dpp(my_lds[(size_t)e * kWave + lane]);
            if (lane == 0 && v != 0.f) unsafeAtomicAdd(&grad_row(E)[(size_t)(E.media_base) * 6 + e], v);
        }
    }
    flush_stats(E, ls);
}

// The instance of a batched plan that owns a tile (wave-uniform).
__device__ __forceinline__ const InstanceDev& tile_instance(const InstanceDev* inst, int n_inst, int64_t tile) {
    int lo_i = 0, hi_i = n_inst - 1;
    while (lo_i < hi_i) {
        const int mid = (lo_i + hi_i + 1) >> 1;
        if (inst[mid].tile_begin <= tile) lo_i = mid; else hi_i = mid - 1;
    }
    return inst[lo_i];
}

// The arguments of an instance's tiles.
template <int EST>
__device__ __forceinline__ EvalArgs instance_args(const EvalArgs& A, const InstanceDev& I) {
    EvalArgs B = A;
    B.root = uni(EST == kEstPhotons ? I.ph_root : I.bm_root);
    B.origin = uni_global(I.origin);
    B.direction = uni_global(I.direction);
    B.offsets = uni_global(I.offsets);
    B.segments = uni_global(I.segments);
    B.perm = I.perm ? uni_global(I.perm) : nullptr;
    B.count = uni64(I.count);
    B.short_query = (int32_t)uni((uint32_t)(I.beam_type == UPBP_SHORT_BEAM));
    B.lite = (int32_t)uni(I.lite);
    B.media_base = (int32_t)uni((uint32_t)I.media_base);
    // an instance's media are the table entries from media_base on: run_tile bounds every
    // instance-local medium id by this count (<= 0 rejects every segment)
    B.n_media = A.n_media - B.media_base;
    B.out = uni_global(EST == kEstPhotons ? I.out_photons : I.out_beams);
    return B;
}

// Persistent batched kernel: waves take (instance, tile) items, or a plan's tasks, from a device
// counter until the queue drains; every wave exits when an index passes
// their number. Structures come from the plan's merged arrays through the kernel
// argument A (wave-uniform scalar loads, see uniform_at); only the instance's root
// node, query pointers and flags come from the instance table. Whole tiles of a plan are gathered like
// those of a launch without one: testing every node for a part of the items cost batches of rays without
// a common origin 8 %. Six waves per SIMD
// (at most 80 VGPRs) measured faster than the unconstrained allocation, and no more: the beam kernel's
// blocks take the registers that the photon kernel's leave and hold them to the end, and with blocks of
// 72 registers before blocks of 80 a quarter of them never found room.
template <int EST, bool PLAN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6, 6))) void k_eval_batched(EvalArgs A, const InstanceDev* __restrict__ inst,
                                                            int n_inst, int64_t total_tiles, uint32_t* queue) {
    constexpr int kMode = (int)Mode::Forward | kBatch;
    const int lane = threadIdx.x & (kWave - 1);
    unsigned long long ls[kStatSlots] = {0, 0, 0, 0, 0, 0, 0, 0};
    const int64_t n_items = PLAN ? (int64_t)as_global(A.plan)->n_tasks : total_tiles;
    while (true) {
        uint32_t item = 0;
        if (lane == 0) item = atomicAdd(queue, 1u);
        item = uni((uint32_t)__shfl(item, 0, kWave));
        if ((int64_t)item >= n_items) break;
        const TileTask t = PLAN ? tile_task(as_global(A.tasks), 0, 0, A.shift, item) : TileTask{item, 0u, 0u, {0u, 0u, 6u}};
        const InstanceDev& I = tile_instance(inst, n_inst, t.tile);
        if (!PLAN) {
            const bool has = EST == kEstPhotons ? I.has_photons : I.has_beams;
            if (!uni((uint32_t)has)) continue;
        }
        const EvalArgs B = instance_args<EST>(A, I);
        const int64_t tile_begin = uni64(I.tile_begin);
        const int64_t slot0 = ((int64_t)t.tile - tile_begin) * kWave;
        if (!PLAN || t.log_parts == 0) {
            run_tile<EST, kMode, false>(B, slot0, t.part, ls, nullptr);
            continue;
        }
        run_tile<EST, kMode | kSplit, false>(B, slot0, t.part, ls, nullptr);
        const TileTask u = tile_task(as_global(A.tasks), 0, 0, A.shift, item);
        if (((int64_t)u.tile - tile_begin) * kWave + lane < B.count)
            for (int c = 0; c < 3; ++c)
                as_global(A.rows)[((size_t)u.row * 3 + c) * kWave + lane] = g_part[threadIdx.x / kWave][c][lane];
    }
    flush_stats(A, ls);
}

// Rebases one instance's copied nodes into the merged array.
__global__ void k_rebase_nodes(NodeDev* nodes, int64_t n, uint32_t node_off, uint32_t item_off) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    uint4 r = nodes[i].r;
    if (r.z != kInvalid) r.x += (r.z & kInner) ? node_off : item_off;
    if (r.w != kInvalid) r.y += (r.w & kInner) ? node_off : item_off;
    nodes[i].r = r;
}

// Adds up the rows of split tiles in the order of their parts: one block per tile, whose waves take
// every fourth row. Row 0 of the grid's y is the photons', row 1 the beams' (null out: nothing to add).
template <class T>
struct SumRows {
    const uint2* info;  // a planned tile's {log2 of its parts, first row}
    uint32_t log_parts;
    const T* rows;
    T* out;
};
template <class T, int N>
__global__ __launch_bounds__(256) void k_sum_rows(int64_t n, const uint32_t* __restrict__ perm, SumRows<T> a,
                                                  SumRows<T> b) {
    __shared__ T part[4][N][kWave];
    const SumRows<T> s = blockIdx.y ? b : a;
    if (!s.out) return;
    const uint32_t tile = blockIdx.x;
    const uint2 info = s.info ? s.info[tile] : make_uint2(s.log_parts, tile << s.log_parts);
    if (info.x == 0) return;  // written by its wave
    const int w = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    const int64_t slot = (int64_t)tile * kWave + lane;
    T v[N] = {};
    if (slot < n)
        for (uint32_t k = w; k < (1u << info.x); k += 4)
            for (int c = 0; c < N; ++c) v[c] += s.rows[((size_t)(info.y + k) * N + c) * kWave + lane];
    for (int c = 0; c < N; ++c) part[w][c][lane] = v[c];
    __syncthreads();
    if (w < N && slot < n)
        s.out[N * (perm ? (int64_t)perm[slot] : slot) + w] =
            ((part[0][w][lane] + part[1][w][lane]) + part[2][w][lane]) + part[3][w][lane];
}

// The same for a batched plan's tiles, whose outputs are their instances': a wave per tile, as most tiles
// have nothing to add.
__global__ __launch_bounds__(256) void k_sum_rows_batched(const InstanceDev* __restrict__ inst, int n_inst, int64_t tiles,
                                                          bool beams, const uint2* __restrict__ infos,
                                                          const float* __restrict__ rows) {
    const uint32_t tile = uni(blockIdx.x * 4u + threadIdx.x / kWave);
    if (tile >= tiles) return;
    const uint2 info = infos[tile];
    if (info.x == 0) return;
    const InstanceDev& I = tile_instance(inst, n_inst, tile);
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t slot = ((int64_t)tile - I.tile_begin) * kWave + lane;
    if (slot >= I.count) return;
    float v[3] = {};
    for (uint32_t k = 0; k < (1u << info.x); ++k)
        for (int c = 0; c < 3; ++c) v[c] += rows[((size_t)(info.y + k) * 3 + c) * kWave + lane];
    float* out = (beams ? I.out_beams : I.out_photons) + 3 * (I.perm ? (int64_t)I.perm[slot] : slot);
    for (int c = 0; c < 3; ++c) out[c] = v[c];
}

// ---- tile plans ----------------------------------------------------------------
// What a tile costs is estimated before a split launch, so that expensive tiles are split into more parts
// than cheap ones and start first. Parts of equal number left a launch waiting for a few waves: of
// 640x360 rays on traced beams the longest wave took 5.8 ms, 20 times the average.
//
// Estimate, one wave per tile: the subtrees of at most frustum_leaf items whose boxes meet the cone
// around the tile's rays within the segments that scatter, 64 nodes at a time (a lane tests a node, where
// the gather tests one node with all rays), weighed as the gather's instruction counts are. Nothing but
// the order and the number of the parts depends on it.
constexpr uint32_t kNoTask = 64;
struct PlanArgs {
    int64_t tiles;
    uint32_t waves, log_most, log_other;  // log_other: of tiles without an estimate
    bool other_apart;                     // those are another launch's, with their rows after the plan's
    uint32_t* cost;
    uint2* info;  // {log2 of the parts, first row}; first the most parts, then the parts and the bucket
    uint2* tasks;
    PlanWords* words;
};

constexpr int kCostQueue = 1024;  // nodes that wait; what does not fit counts without being opened,
// as does what is left after kCostSteps steps, or a 128th of the tiles: a launch of more tiles takes longer
// and can wait longer for its plan. With 64 steps the tiles next to a light counted for too little and one
// of their waves took 31 ms of 1920x1080 rays on 125k traced beams (35.2 ms, 23.1 with 256).
constexpr int kCostSteps = 256;
constexpr uint32_t kCostNone = 0;             // a tile with nothing to gather

template <int EST>
__device__ __forceinline__ float tile_cost(const EvalArgs& A, int64_t slot, int steps, uint32_t group, uint32_t* nodes,
                                           bool& one) {
    constexpr float kNode = 46.f, kLeaf = 73.f, kItem = EST == kEstPhotons ? 8.f : 20.f, kTile = 500.f;
    const int lane = threadIdx.x & (kWave - 1);
    const QueryIn in = read_query(A, slot);
    const float dx = in.d[0], dy = in.d[1], dz = in.d[2];
    float t0 = __builtin_inff(), t1 = -__builtin_inff();
    if (in.alive)
        for (int64_t k = in.s0; k < in.s0 + in.nseg; ++k) {
            const upbp_volume_segment* sg = A.segments + k;
            const int32_t m = sg->medium_id;
            if (m < 0 || m >= A.n_media) break;
            if (A.media[A.media_base + m].has_scattering) {
                t0 = fminf(t0, sg->dist_min);
                t1 = fmaxf(t1, sg->dist_max);
            }
        }
    const uint64_t am = __ballot(t0 <= t1);
    float c = 0.f;
    one = common_origin(A, in);
    if (am) {
        const int fl = __builtin_ctzll(am);
        const bool on = t0 <= t1;
        const float px = __shfl(in.o[0], fl, kWave), py = __shfl(in.o[1], fl, kWave), pz = __shfl(in.o[2], fl, kWave);
        const float len = __builtin_sqrtf((dx * dx + dy * dy) + dz * dz);
        const float il = on && len > 0.f ? 1.f / len : 0.f;
        const float ux = dx * il, uy = dy * il, uz = dz * il;
        float ax = ux, ay = uy, az = uz, lo = on ? t0 * len : __builtin_inff(), hi = on ? t1 * len : 0.f;
        for (int off = 32; off > 0; off >>= 1) {
            ax += __shfl_xor(ax, off, kWave);
            ay += __shfl_xor(ay, off, kWave);
            az += __shfl_xor(az, off, kWave);
            lo = fminf(lo, __shfl_xor(lo, off, kWave));
            hi = fmaxf(hi, __shfl_xor(hi, off, kWave));
        }
        const float al = __builtin_sqrtf((ax * ax + ay * ay) + az * az);
        const float ia = al > 0.f ? 1.f / al : 0.f;
        ax *= ia, ay *= ia, az *= ia;
        float cs = on ? (ux * ax + uy * ay) + uz * az : 1.f;
        for (int off = 32; off > 0; off >>= 1) cs = fminf(cs, __shfl_xor(cs, off, kWave));
        const float tn = cs > 0.1f ? __builtin_sqrtf(fmaxf(1.f - cs * cs, 0.f)) / cs : 10.f;
        const float ix = guard_inv(ax), iy = guard_inv(ay), iz = guard_inv(az);
        int head = 0, size = one ? 1 : 0;
        if (lane == 0) nodes[0] = A.root;
        for (int step = 0; size > 0; ++step) {
            wave_lds_sync();
            // the oldest nodes, or the newest (fewer new ones) where the queue could overflow
            const int n = min(size, kWave);
            const bool newest = size > kCostQueue - 2 * kWave;
            const int from = newest ? head + size - n : head;
            if (!newest) head = (head + n) % kCostQueue;
            size -= n;
            bool go[2] = {false, false};
            uint32_t ref[2] = {0u, 0u};
            float skipped[2] = {0.f, 0.f};
            if (lane < n) {
                const NodeDev nd = A.nodes[nodes[(from + lane) % kCostQueue]];
                const float bl[2][3] = {{nd.a.x, nd.a.y, nd.a.z}, {nd.b.z, nd.b.w, nd.c.x}};
                const float bh[2][3] = {{nd.a.w, nd.b.x, nd.b.y}, {nd.c.y, nd.c.z, nd.c.w}};
                const uint32_t kind[2] = {nd.r.z, nd.r.w};
                ref[0] = nd.r.x, ref[1] = nd.r.y;
                c += kNode;
                for (int k = 0; k < 2; ++k) {
                    if (kind[k] == kInvalid) continue;
                    // the axis against the box, widened by the cone's radius at the box's far side
                    const float mx = 0.5f * (bl[k][0] + bh[k][0]) - px, my = 0.5f * (bl[k][1] + bh[k][1]) - py,
                                mz = 0.5f * (bl[k][2] + bh[k][2]) - pz;
                    const float hx = 0.5f * (bh[k][0] - bl[k][0]), hy = 0.5f * (bh[k][1] - bl[k][1]),
                                hz = 0.5f * (bh[k][2] - bl[k][2]);
                    const float rad = __builtin_amdgcn_sqrtf((hx * hx + hy * hy) + hz * hz);
                    const float far = __builtin_amdgcn_sqrtf((mx * mx + my * my) + mz * mz) + rad;
                    const float e = fmaxf(tn * fminf(far, hi), 1e-30f);
                    const float wx = (hx + e) * __builtin_fabsf(ix), wy = (hy + e) * __builtin_fabsf(iy),
                                wz = (hz + e) * __builtin_fabsf(iz);
                    const float cx = mx * ix, cy = my * iy, cz = mz * iz;
                    const float near = fmaxf(fmaxf(cx - wx, cy - wy), fmaxf(cz - wz, lo));
                    const float past = fminf(fminf(cx + wx, cy + wy), fminf(cz + wz, hi));
                    if (!(near <= past)) continue;
                    const uint32_t items = kind[k] & kSpanMask;
                    float cost = kLeaf + (kLeaf / 64.f + kItem) * (float)items;
                    if ((kind[k] & kInner) && items > 64u) {
                        // of a larger subtree, the runs of 64 items that the cone crosses
                        const float part = __builtin_amdgcn_exp2f(
                            __builtin_amdgcn_logf(64.f / (float)items) * (1.f / 3.f));
                        const float f = (e + part * rad) * __builtin_amdgcn_rcpf(e + rad);
                        cost *= f * f;
                        go[k] = items > group && step < steps;
                    }
                    if (go[k])
                        skipped[k] = cost;
                    else
                        c += cost;
                }
            }
            wave_lds_sync();  // the popped entries are read before others take their place
            for (int k = 0; k < 2; ++k) {
                const uint64_t m = __ballot(go[k]);
                const int at = size + __builtin_popcountll(m & ((1ull << lane) - 1ull));
                if (go[k]) {
                    if (at < kCostQueue)
                        nodes[(head + at) % kCostQueue] = ref[k];
                    else
                        c += skipped[k];
                }
                size = min(size + __builtin_popcountll(m), kCostQueue);
            }
        }
    }
    for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, kWave);
    return c + kTile;
}

// Writes a tile's cost and the most parts it may have (log2), and adds it to the total.
__device__ __forceinline__ void put_cost(const PlanArgs& P, uint32_t tile, float c, bool one, uint32_t log_most) {
    if ((threadIdx.x & (kWave - 1)) != 0) return;
    const uint32_t v = (uint32_t)fminf(c, 4e9f);
    P.cost[tile] = one ? v : kCostOther;
    P.info[tile] = make_uint2(one ? log_most : P.log_other, 0u);
    if (one) {
        atomicAdd(&P.words->total[blockIdx.x % 64][0], (unsigned long long)v);
        atomicAdd(&P.words->total[blockIdx.x % 64][1], 1ull);
    }
}

template <int EST>
__global__ __launch_bounds__(256) void k_tile_cost(EvalArgs A, PlanArgs P, int steps) {
    __shared__ uint32_t queue[4][kCostQueue];
    const uint32_t tile = uni(blockIdx.x * 4u + threadIdx.x / kWave);
    if (tile >= P.tiles) return;
    bool one;
    const float c = tile_cost<EST>(A, (int64_t)tile * kWave + (threadIdx.x & (kWave - 1)), steps,
                                   A.frustum_leaf, queue[threadIdx.x / kWave], one);
    put_cost(P, tile, c, one, P.log_most);
}

// The same over the tiles of a batched plan's instances, of which there are many: one estimate, from every
// kBatchStride-th ray, for kBatchStride consecutive tiles of an instance.
constexpr int kBatchStride = 16, kBatchSteps = 16;
template <int EST>
__global__ __launch_bounds__(256) void k_tile_cost_batched(EvalArgs A, PlanArgs P, const InstanceDev* __restrict__ inst, int n_inst) {
    __shared__ uint32_t queue[4][kCostQueue];
    const uint32_t tile = uni(blockIdx.x * 4u + threadIdx.x / kWave);
    if (tile >= P.tiles) return;
    const InstanceDev& I = tile_instance(inst, n_inst, tile);
    if (!uni((uint32_t)(EST == kEstPhotons ? I.has_photons : I.has_beams))) {
        if ((threadIdx.x & (kWave - 1)) == 0) P.cost[tile] = kCostNone;
        return;
    }
    const int64_t local = (int64_t)tile - uni64(I.tile_begin);
    if (local % kBatchStride != 0) return;
    const EvalArgs B = instance_args<EST>(A, I);
    bool one;
    const float c = tile_cost<EST>(B, local * kWave + (threadIdx.x & (kWave - 1)) * kBatchStride, kBatchSteps,
                                   uni(EST == kEstPhotons ? I.ph_group : I.bm_group), queue[threadIdx.x / kWave], one);
    const int64_t tiles = (B.count + kWave - 1) / kWave;
    for (int k = 0; k < kBatchStride && local + k < tiles; ++k)
        put_cost(P, tile + k, c, one, uni(EST == kEstPhotons ? I.ph_log_most : I.bm_log_most));
}

// Parts per tile: the share of `waves` that its cost is of the whole, rounded down to a power of two, so
// that all parts together are no more than `waves`. Then a counting sort of the parts by what one costs,
// in quarter octaves, dearest first.

__global__ __launch_bounds__(256) void k_plan_parts(PlanArgs P) {
    __shared__ uint32_t hist[64];
    __shared__ float share;
    if (threadIdx.x < 64) {
        hist[threadIdx.x] = 0;
        unsigned long long t = P.words->total[threadIdx.x][0], n = P.words->total[threadIdx.x][1];
        for (int off = 32; off > 0; off >>= 1) {
            t += __shfl_xor(t, off, kWave);
            n += __shfl_xor(n, off, kWave);
        }
        if (threadIdx.x == 0)
            share = (float)((double)P.waves * (double)n / ((double)P.tiles * (double)(t > 0 ? t : 1)));
    }
    __syncthreads();
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < P.tiles) {
        const uint32_t c = P.cost[i];
        const uint32_t most = P.info[i].x;
        uint32_t lg = most, bucket = 0;
        if (c == kCostNone) {
            lg = 0;
            bucket = kNoTask;
        } else if (c != kCostOther) {
            const float want = (float)c * share;
            lg = 0;
            while (lg < most && want >= (float)(2u << lg)) ++lg;
            const int q = (int)(__float_as_uint(want / (float)(1u << lg)) >> 21) - (int)(__float_as_uint(1.f) >> 21);
            bucket = (uint32_t)min(max(24 - q, 0), 63);
        }
        if (c == kCostOther && P.other_apart) bucket = kNoTask;
        P.info[i] = make_uint2(lg, bucket);
        if (bucket != kNoTask) atomicAdd(&hist[bucket], 1u << lg);
    }
    __syncthreads();
    if (threadIdx.x < 64 && hist[threadIdx.x]) atomicAdd(&P.words->hist[threadIdx.x], hist[threadIdx.x]);
}

__global__ __launch_bounds__(256) void k_plan_tasks(PlanArgs P) {
    __shared__ uint32_t base[64], taken[64], rows, row_base;
    if (threadIdx.x < 64) {
        const uint32_t h = P.words->hist[threadIdx.x];
        uint32_t x = h;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y = __shfl_up(x, off, kWave);
            x += (int)threadIdx.x >= off ? y : 0u;
        }
        base[threadIdx.x] = x - h;
        taken[threadIdx.x] = 0;
        if (threadIdx.x == 63 && blockIdx.x == 0) P.words->n_tasks = x;
        if (threadIdx.x == 0) rows = 0;
    }
    __syncthreads();
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    uint2 info = make_uint2(0u, kNoTask);
    uint32_t at = 0, row = 0;
    if (i < P.tiles) info = P.info[i];
    if (info.y != kNoTask) {
        at = atomicAdd(&taken[info.y], 1u << info.x);
        if (info.x) row = atomicAdd(&rows, 1u << info.x);
    }
    __syncthreads();
    if (threadIdx.x < 64 && taken[threadIdx.x])
        base[threadIdx.x] += atomicAdd(&P.words->cursor[threadIdx.x], taken[threadIdx.x]);
    if (threadIdx.x == 64) row_base = atomicAdd(&P.words->n_rows, rows);
    __syncthreads();
    const bool task = info.y != kNoTask;
    at += task ? base[info.y] : 0u;
    row = task ? row + row_base : P.waves + ((uint32_t)i << info.x);
    if (i < P.tiles) P.info[i] = make_uint2(info.x, row);
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t first = (uint32_t)(i - lane);
    for (uint64_t m = __ballot(task); m; m &= m - 1) {  // the wave writes each tile's tasks together
        const int k = __builtin_ctzll(m);
        const uint32_t lg = __shfl(info.x, k, kWave), to = __shfl(at, k, kWave), r = __shfl(row, k, kWave);
        for (uint32_t j = lane; j < (1u << lg); j += kWave)
            P.tasks[to + j] =
                make_uint2(first + k, j | (lg << kTaskPartBits) | ((r + j) << (kTaskPartBits + kTaskLogBits)));
    }
}

__global__ void k_clear_u64(unsigned long long* p, int64_t n) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}
__global__ void k_clear_f32(float* p, int64_t n) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.f;
}
__global__ void k_fill_u32(uint32_t* p, uint32_t v, int64_t n) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_combine_media(const float* gm, int rows, const float* sign, int n, float* gs, float* ga) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 3 * n) return;
    const int m = i / 3, c = i % 3;
    float direct = 0.f, dt = 0.f;
    for (int r = 0; r < rows; ++r) {
        direct += gm[6 * ((size_t)r * n + m) + c];
        dt += gm[6 * ((size_t)r * n + m) + 3 + c];
    }
    if (gs) gs[i] += sign[6 * m + 3 + c] * (direct + dt);
    if (ga) ga[i] += sign[6 * m + c] * dt;
}

// Distance along the 15-bit Hilbert curve of the cell (x, y), in 30 bits.
__device__ __forceinline__ uint32_t hilbert2(uint32_t x, uint32_t y) {
    uint32_t d = 0;
    for (int b = 14; b >= 0; --b) {
        const uint32_t rx = (x >> b) & 1u, ry = (y >> b) & 1u;
        d = (d << 2) | ((3u * rx) ^ ry);
        const uint32_t low = (1u << b) - 1u;
        x &= low;
        y &= low;
        if (!ry) {
            const uint32_t f = rx ? low : 0u;  // reflected, then transposed
            const uint32_t t = x ^ f;
            x = y ^ f;
            y = t;
        }
    }
    return d;
}

constexpr uint32_t kOtherOrigin = 1u << (kQueryKeyBits - 1);  // key bit of the queries that do not start at query 0's origin

// Sort key of a query, so that consecutive lanes hold coherent queries: the Morton code of its
// first segment's entry point, or with by_direction
//  - for a query from query 0's origin (the camera rays of a frame) its direction alone: the place
//    on the octahedral map, turned so that query 0's main axis is the map's centre (the map's seam
//    then lies opposite), along a Hilbert curve. 64 consecutive cells of that curve are one connected
//    patch, so a wave's frustum is small wherever its run of 64 starts, while a run of the Morton
//    order jumps: on 1920x1080 rays the frusta span 0.0055 x 0.0081 of the z = 0 plane on average
//    in Morton order, 0.0045 x 0.0045 here (8 x 8 tiles: 0.0036 x 0.0036). The segments are not read.
//  - for the others, after those, the Morton code.
// Only evaluations without beams go by direction (256x256 rays x 100k photons: 402 -> 295 us). A beam's
// end ties (test_beam_beam) are found where the wave's other rays visit the leaf, so which of them are
// found depends on the rays that share a wave: beams keep the one order, and with it the same hits.
__global__ void k_query_keys(int64_t n, const float* __restrict__ origin, const float* __restrict__ direction,
                             const int64_t* __restrict__ offsets, const upbp_volume_segment* __restrict__ seg,
                             float lx, float ly, float lz, float sx, float sy, float sz,
                             bool by_direction, uint32_t* keys, uint32_t* idx) {
    int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (q >= n) return;
    idx[q] = (uint32_t)q;
    const float ox = origin[3 * q], oy = origin[3 * q + 1], oz = origin[3 * q + 2];
    const float dx = direction[3 * q], dy = direction[3 * q + 1], dz = direction[3 * q + 2];
    if (by_direction && ox == origin[0] && oy == origin[1] && oz == origin[2]) {
        const float ax = __builtin_fabsf(direction[0]), ay = __builtin_fabsf(direction[1]),
                    az = __builtin_fabsf(direction[2]);
        float u = dx, v = dy, w = dz, s = direction[2];  // w: along query 0's main axis
        if (ax >= ay && ax >= az)
            u = dy, v = dz, w = dx, s = direction[0];
        else if (ay >= az)
            u = dz, v = dx, w = dy, s = direction[1];
        w = s < 0.f ? -w : w;
        const float l1 = (__builtin_fabsf(u) + __builtin_fabsf(v)) + __builtin_fabsf(w);
        u /= l1, v /= l1;
        if (w < 0.f) {
            const float fu = 1.f - __builtin_fabsf(v), fv = 1.f - __builtin_fabsf(u);
            u = u < 0.f ? -fu : fu;
            v = v < 0.f ? -fv : fv;
        }
        // a zero or non-finite direction maps to cell 0: the evaluation reports it
        const float cu = fminf(fmaxf((u + 1.f) * 16384.f, 0.f), 32767.f),
                    cv = fminf(fmaxf((v + 1.f) * 16384.f, 0.f), 32767.f);
        keys[q] = hilbert2((uint32_t)cu, (uint32_t)cv);
        return;
    }
    const int64_t s0 = offsets[q], s1 = offsets[q + 1], sn = offsets[n];
    float t = 0.f;
    // first segment in a scattering-capable position: use its start
    if (s0 >= 0 && s0 < s1 && s1 <= sn) {
        const int64_t last = s1 - 1;
        t = seg[s0].dist_min;
        // skip a leading clear segment (camera outside the media) when there is a next one
        if (s0 < last) t = seg[s0 + 1].dist_min;
    }
    float p[3] = {ox + dx * t, oy + dy * t, oz + dz * t};
    const float l[3] = {lx, ly, lz}, s[3] = {sx, sy, sz};
    uint32_t key = 0;
    uint32_t c[3];
    for (int a = 0; a < 3; ++a) {
        float u = (p[a] - l[a]) * s[a];
        u = __builtin_isfinite(u) ? fminf(fmaxf(u, 0.f), 1023.f) : 0.f;
        c[a] = (uint32_t)u;
    }
    for (int b = 9; b >= 0; --b)
        key = (key << 3) | (((c[0] >> b) & 1u) << 2) | (((c[1] >> b) & 1u) << 1) | ((c[2] >> b) & 1u);
    keys[q] = by_direction ? kOtherOrigin | key : key;
}

inline unsigned grid_for(int64_t n, int block = 256) {
    return (unsigned)std::max<int64_t>(1, (n + block - 1) / block);
}

// 2^shift items per block of a split, 64 or more (ItemPart::items): 32 to 64 blocks per part where there
// are enough. Fewer balance worse (8: 22.0 against 20.0 ms on 200k rays without a common origin, 7.9
// against 7.0 ms on traced beams), more make every part walk more of the tree.
static uint32_t part_shift(int64_t items) {
    uint32_t shift = 0;
    while (((int64_t)32 << (shift + 1)) <= items) ++shift;
    return shift;
}

// A block of one wave gives its place up as soon as that wave ends: with 1 / 2 / 4 waves of a plan per block
// 1M rays on 2M beams take 36.7 / 38.0 / 38.7 ms, 1920x1080 rays 8.57 / 8.67 / 8.81 ms (adjoint blocks keep 4).
constexpr int kTaskWaves = 1;
template <int EST, int MODE>
void launch_waves(Ctx& ctx, const EvalArgs& A, int64_t waves, int tuned) {
    // the tuned number of waves per block, one of a plan's tasks, or up to 4 parts of one tile
    const bool adjoint = (MODE & 7) == (int)Mode::Adjoint;
    const int wpb = A.tasks && !adjoint                    ? kTaskWaves
                    : A.tasks || (adjoint && A.log_parts == 0) ? 4
                    : A.log_parts > 0                        ? std::min(1 << A.log_parts, 4)
                                                             : std::min(std::max(tuned, 1), 4);
    const dim3 blocks((unsigned)((waves + wpb - 1) / wpb)), threads((unsigned)(wpb * kWave));
    // LDS gradient slabs for the media actually present: fewer bytes, more resident waves
    const size_t lds = adjoint ? (size_t)wpb * A.lds_media_n * 6 * kWave * sizeof(float) : 0;
    if (A.tasks || A.log_parts > 0)
        hipLaunchKernelGGL((k_eval<EST, MODE | kSplit>), blocks, threads, lds, ctx.stream, A);
    else
        hipLaunchKernelGGL((k_eval<EST, MODE>), blocks, threads, lds, ctx.stream, A);
    UPBP_HIP(hipGetLastError());
}

static int cost_steps(int64_t tiles) { return (int)std::min<int64_t>(std::max<int64_t>(tiles / 128, 16), kCostSteps); }

static void launch_plan(Ctx& ctx, const PlanArgs& P) {
    hipLaunchKernelGGL(k_plan_parts, dim3(grid_for(P.tiles)), dim3(256), 0, ctx.stream, P);
    hipLaunchKernelGGL(k_plan_tasks, dim3(grid_for(P.tiles)), dim3(256), 0, ctx.stream, P);
    UPBP_HIP(hipGetLastError());
}

// An evaluation's launches, with its split set up. A plan gives the tiles with a common origin their parts;
// the others are split uniformly.
template <int EST, int MODE>
void launch_kernel(Ctx& ctx, EvalArgs A, const Split& s, const TilePlan& p, int64_t items, int tuned) {
    // one ray has one origin; few pieces take less time than a second launch
    const bool two = A.count > 1 && (EST == kEstPhotons || items >= kSparseFrom);
    const int64_t tiles = (A.count + kWave - 1) / kWave;
    A.known = s.planned || !two;
    if (s.planned) {
        EvalArgs B = A;
        B.tasks = p.tasks;
        B.plan = p.words;
        const PlanArgs P = {tiles, (uint32_t)s.waves, s.log_most, s.log_parts, in_two(MODE), p.cost, p.info, p.tasks, p.words};
        const int steps = cost_steps(tiles);
        hipLaunchKernelGGL(k_tile_cost<EST>, dim3(grid_for(tiles, 4)), dim3(256), 0, ctx.stream, B, P, steps);
        launch_plan(ctx, P);
        launch_waves<EST, MODE>(ctx, B, tiles + s.waves, tuned);
        A.row0 = (uint32_t)s.waves;
        A.tile_class = p.cost;
    } else {
        launch_waves<EST, MODE>(ctx, A, tiles << s.log_parts, tuned);
    }
    if constexpr (in_two(MODE))
        if (two) launch_waves<EST, MODE | kSparse>(ctx, A, tiles << s.log_parts, tuned);
}

template <int EST, int MODE>
void launch_reduced(Ctx& ctx, const EvalArgs& A, const Split& s, const TilePlan& p, int64_t items, int tuned) {
    if constexpr (EST == kEstBeams) {
        if (A.red.max != 0) return launch_kernel<EST, MODE | kReduced>(ctx, A, s, p, items, tuned);
    }
    launch_kernel<EST, MODE>(ctx, A, s, p, items, tuned);
}

template <int EST>
void launch_mode(Ctx& ctx, Mode mode, EvalArgs& A, const QueryView& q, int64_t items, int tuned) {
    const Split& s = q.split[EST];
    const TilePlan& p = q.plan[EST];
    A.log_parts = s.log_parts;
    A.shift = part_shift(items);
    A.rows = p.rows;
    switch (mode) {
        case Mode::Forward: return launch_reduced<EST, (int)Mode::Forward>(ctx, A, s, p, items, tuned);
        case Mode::Signature: return launch_reduced<EST, (int)Mode::Signature>(ctx, A, s, p, items, tuned);
        case Mode::Adjoint: return launch_reduced<EST, (int)Mode::Adjoint>(ctx, A, s, p, items, tuned);
        case Mode::Upbp: return launch_reduced<EST, (int)Mode::Upbp>(ctx, A, s, p, items, tuned);
    }
}

EvalArgs base_args(Ctx& ctx, const QueryView& q) {
    EvalArgs A = {};
    A.origin = q.origin;
    A.direction = q.direction;
    A.offsets = q.offsets;
    A.segments = q.segments;
    A.perm = q.perm;
    A.count = q.count;
    A.short_query = q.beam_type == UPBP_SHORT_BEAM;
    A.lite = (int32_t)q.lite;
    A.media = ctx.media.as<MediumDev>();
    A.n_media = ctx.n_media;
    A.media_base = 0;
    A.lds_media_n = std::max(1, std::min(ctx.n_media, kMaxLdsMedia));
    A.stats = ctx.stats.as<unsigned long long>();
    A.frustum_leaf = (uint32_t)ctx.tuning.frustum_leaf;
    return A;
}

}  // namespace

// The tail of every light vertex. A chain is a vertex of path length 0 and those after it whose stored
// path lengths count 1, 2, ...; each vertex's terms are folded into the tail of the next one, and a vertex
// no chain reaches gets the NaN below-marker. A block reads 256 consecutive vertices once, a thread each,
// and the chains are walked in LDS by the threads of their first vertices; thread 0 first walks the part of
// its chain that lies before the block. Bound by the reads (112 bytes per vertex). A thread per chain that
// walked it in memory took 228 us on 3.5M vertices, with a separate launch for the markers; this takes 118.
constexpr int kTailBlock = 256;
struct TailTerms {
    float t_rest, t_ray, b, rev, ray_rev, inv;
};
__device__ __forceinline__ TailTerms tail_terms(const upbp_mis_data& d, bool next_spec, const upbp_mis_params& p) {
    TailTerms t;
    light_tail_terms(d, p.techniques, p.query_beam_type, p.photon_beam_type, t.t_rest, t.t_ray);
    const bool spec = (d.flags & UPBP_MIS_SPECULAR) != 0;
    t.b = ((p.techniques & UPBP_BPT) && !spec && !next_spec) ? 1.f : 0.f;
    t.rev = d.rev_pdf_a;
    t.ray_rev = d.ray_sample_rev_pdf_inv;
    t.inv = d.pdf_a_inv;
    return t;
}
__device__ __forceinline__ float tail_below(const TailTerms& t, float below) {
    return t.rev == 0.f ? 0.f : t.rev * ((t.t_rest + t.ray_rev * t.t_ray) + t.inv * (t.b + below));
}

__global__ __launch_bounds__(kTailBlock) void k_light_tails(const upbp_light_vertex* __restrict__ lv, int64_t n,
                                                            upbp_mis_params p, float4* __restrict__ tails) {
    __shared__ TailTerms terms[kTailBlock];
    __shared__ float below[kTailBlock];
    __shared__ uint32_t length[kTailBlock];
    __shared__ bool reached[kTailBlock];
    const int64_t base = (int64_t)blockIdx.x * kTailBlock, m = base + threadIdx.x;
    const int here = (int)min((int64_t)kTailBlock, n - base);
    const auto specular = [&](int64_t v) { return (lv[v].mis.flags & UPBP_MIS_SPECULAR) != 0; };
    below[threadIdx.x] = __builtin_nanf("");
    reached[threadIdx.x] = false;
    if (m < n) {
        length[threadIdx.x] = lv[m].path_length;
        // a chain's first vertex has no next one: its own flag stands for it
        terms[threadIdx.x] = tail_terms(lv[m].mis, specular(lv[m].path_length > 0 && m > 0 ? m - 1 : m), p);
    }
    __syncthreads();
    const uint32_t len = m < n ? length[threadIdx.x] : 1u;
    bool walks = len == 0;
    float x = 0.f;  // tail of the vertex under the current one
    if (threadIdx.x == 0 && len > 0 && (int64_t)len <= base) {
        const int64_t s = base - len;
        walks = true;
        for (int64_t v = s; v < base && walks; ++v) {
            walks = lv[v].path_length == (uint32_t)(v - s);
            x = tail_below(tail_terms(lv[v].mis, specular(v > s ? v - 1 : v), p), x);
        }
    }
    if (walks)
        for (int k = threadIdx.x; k < here && length[k] == len + (uint32_t)(k - threadIdx.x); ++k) {
            below[k] = x;
            reached[k] = true;
            x = tail_below(terms[k], x);
        }
    __syncthreads();
    if (m >= n) return;
    const TailTerms t = terms[threadIdx.x];
    const float u = below[threadIdx.x];
    tails[m] = reached[threadIdx.x] ? make_float4(t.t_rest, t.t_ray, t.b, u) : make_float4(0.f, 0.f, 0.f, u);
}

__global__ void k_beam_records(MisGlobals G, int64_t n, BeamRec* __restrict__ out) {
    const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= n) return;
    const upbp_beam_mis bm = G.beams[b];
    BeamRec r = {};
    r.light_vertex = bm.light_vertex;
    if (bm.light_vertex < 0 || (int64_t)bm.light_vertex >= G.lv_count) {
        r.info = kRecBadVertex;
        out[b] = r;
        return;
    }
    const upbp_light_vertex* __restrict__ lv = G.lv + bm.light_vertex;
    r.tail = G.tails ? G.tails[bm.light_vertex] : make_float4(0.f, 0.f, 0.f, __builtin_nanf(""));
    r.ray_sample_pdf = bm.ray_sample_pdf;
    r.ray_sample_rev_pdf = bm.ray_sample_rev_pdf;
    r.last_pdf_w_inv = bm.last_pdf_w_inv;
    r.cos_theta_out = lv->mis.cos_theta_out;
    r.pdf_a_inv = lv->mis.pdf_a_inv;
    r.lv_flags = lv->mis.flags;
    r.path_idx = lv->path_idx;
    const uint32_t len = lv->path_length;
    // light_weight_tail_bb1d's test that the tails apply: the vertex ends the stored chain
    const bool chain =
        G.tails && light_last_index(G, lv->path_idx, (int)len + 1) == (int64_t)bm.light_vertex + 1;
    r.info = (len < kRecLengthMask ? len : kRecLengthMask) | (lv->is_finite ? kRecFinite : 0u) |
             ((bm.ray_sampling_flags & UPBP_ORIGIN_IN_MEDIUM) ? kRecOriginInMedium : 0u) | (chain ? kRecTailChain : 0u);
    out[b] = r;
}

// light_weight_tail's inputs per light vertex v: everything but `last` and `ntl`.
__global__ void k_photon_records(MisGlobals G, PhotonRec* __restrict__ out) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= G.lv_count) return;
    const upbp_light_vertex* __restrict__ lv = G.lv + v;
    PhotonRec r;
    r.a = make_float4(lv->throughput[0], lv->throughput[1], lv->throughput[2], lv->continuation_prob);
    r.b = make_float4(lv->dir_fix[0], lv->dir_fix[1], lv->dir_fix[2], lv->mis.ray_sample_pdf_inv);
    const uint32_t len = lv->path_length;
    const bool has1 = len > 0;
    uint32_t info = len < kRecLengthMask ? len : kRecLengthMask;
    if (G.tails && light_last_index(G, lv->path_idx, (int)len) == v && v >= (has1 ? 1 : 0)) info |= kPRecChain;
    if (has1) info |= kPRecHas1;
    float cs = 0.f, tt = 0.f;
    if (info & kPRecChain) {
        const upbp_light_vertex* __restrict__ nx = has1 ? lv - 1 : lv;
        if (!(nx->mis.flags & UPBP_MIS_SPECULAR)) info |= kPRecNextPlain;
        if (has1) {
            const float4 t = G.tails[v - 1];
            if (!__builtin_isnan(t.w) && (int)nx->path_length == (int)len - 1) {
                info |= kPRecNextTail;
                cs = nx->mis.rev_pdf_a_without_bsdf;
                tt = (t.x + nx->mis.ray_sample_rev_pdf_inv * t.y) + nx->mis.pdf_a_inv * (t.z + t.w);
            }
        }
    }
    r.c = make_float4(lv->mis.ray_sample_pdfs_ratio, lv->mis.pdf_a_inv, cs, tt);
    r.d = make_uint4(info, (uint32_t)lv->path_idx, (uint32_t)v, 0u);
    out[v] = r;
}

void launch_photon_records(Ctx& ctx, MisDev& mis) {
    mis.photon_recs = nullptr;
    if (mis.lv_count <= 0) return;
    ctx.photon_recs.ensure((size_t)mis.lv_count * sizeof(PhotonRec));
    MisGlobals G = {};
    G.lv = mis.lv;
    G.lv_count = mis.lv_count;
    G.path_ends = mis.path_ends;
    G.path_count = mis.path_count;
    G.p = mis.params;
    G.tails = mis.tails;
    hipLaunchKernelGGL(k_photon_records, dim3(grid_for(mis.lv_count)), dim3(256), 0, ctx.stream, G,
                       ctx.photon_recs.as<PhotonRec>());
    UPBP_HIP(hipGetLastError());
    mis.photon_recs = ctx.photon_recs.p;
}

void launch_beam_records(Ctx& ctx, MisDev& mis, int64_t n_beams) {
    mis.beam_recs = nullptr;
    if (n_beams <= 0 || !mis.beams) return;
    ctx.beam_recs.ensure((size_t)n_beams * sizeof(BeamRec));
    MisGlobals G = {};
    G.lv = mis.lv;
    G.lv_count = mis.lv_count;
    G.path_ends = mis.path_ends;
    G.path_count = mis.path_count;
    G.beams = mis.beams;
    G.p = mis.params;
    G.tails = mis.tails;
    hipLaunchKernelGGL(k_beam_records, dim3(grid_for(n_beams)), dim3(256), 0, ctx.stream, G, n_beams,
                       ctx.beam_recs.as<BeamRec>());
    UPBP_HIP(hipGetLastError());
    mis.beam_recs = ctx.beam_recs.p;
}

void launch_light_tails(Ctx& ctx, MisDev& mis) {
    mis.tails = nullptr;
    if (mis.lv_count <= 0) return;
    ctx.light_tails.ensure((size_t)mis.lv_count * sizeof(float4));
    float4* t = ctx.light_tails.as<float4>();
    hipLaunchKernelGGL(k_light_tails, dim3(grid_for(mis.lv_count, kTailBlock)), dim3(kTailBlock), 0, ctx.stream, mis.lv,
                       mis.lv_count, mis.params, t);
    UPBP_HIP(hipGetLastError());
    mis.tails = t;
}

static void set_mis(EvalArgs& A, const MisDev* mis) {
    if (!mis) return;
    A.mis.tails = mis->tails;
    A.qmis = mis->queries;
    A.mis.camera = mis->camera;
    A.mis.camera_count = mis->camera_count;
    A.mis.lv = mis->lv;
    A.mis.lv_count = mis->lv_count;
    A.mis.path_ends = mis->path_ends;
    A.mis.path_count = mis->path_count;
    A.mis.beams = mis->beams;
    A.mis.beam_recs = static_cast<const BeamRec*>(mis->beam_recs);
    A.mis.photon_recs = static_cast<const PhotonRec*>(mis->photon_recs);
    A.mis.p = mis->params;
}

Split split_of(int64_t count, int64_t items, int est, Mode mode) {
    Split s;
    if (items < kSplitFrom) return s;
    s.tiles = (count + kWave - 1) / kWave;
    const bool light = mode == Mode::Upbp || est == kEstPhotons;
    s.waves = light ? kSplitWavesLight : kSplitWaves;
    const auto fits = [&](uint32_t lg) { return (kSplitItems << lg) <= items; };
    while ((2u << s.log_parts) <= kSplitMost && (s.tiles << (s.log_parts + 1)) <= s.waves && fits(s.log_parts + 1))
        ++s.log_parts;
    s.planned = !light && s.tiles >= kPlanTiles && s.tiles <= kPlanMostTiles;
    if (s.planned) {
        if (s.tiles <= kPlanFewTiles) s.waves = kPlanWaves;
        while ((2u << s.log_most) <= kPlanMost && fits(s.log_most + 1)) ++s.log_most;
    }
    if (mode != Mode::Adjoint)
        s.rows = (s.planned ? s.waves : 0) + (s.log_parts > 0 ? s.tiles << s.log_parts : 0);
    return s;
}

template <class T, int N>
static void sum_rows(Ctx& ctx, const QueryView& q, T* ph, T* bm) {
    SumRows<T> a[2];
    for (int e = 0; e < 2; ++e) {
        const Split& s = q.split[e];
        a[e] = {s.planned ? q.plan[e].info : nullptr, s.log_parts, reinterpret_cast<const T*>(q.plan[e].rows),
                s.rows ? (e == kEstPhotons ? ph : bm) : nullptr};
    }
    if (!a[0].out && !a[1].out) return;
    hipLaunchKernelGGL((k_sum_rows<T, N>), dim3((unsigned)((q.count + kWave - 1) / kWave), 2), dim3(256), 0, ctx.stream,
                       q.count, q.perm, a[0], a[1]);
    UPBP_HIP(hipGetLastError());
}

void launch_sum_rows(Ctx& ctx, const QueryView& q, float* ph, float* bm) { sum_rows<float, 3>(ctx, q, ph, bm); }
void launch_sum_rows_sig(Ctx& ctx, const QueryView& q, uint32_t* ph, uint32_t* bm) {
    sum_rows<uint32_t, 2>(ctx, q, ph, bm);
}

void launch_photons(Ctx& ctx, Mode mode, const PhotonArgs& ph, const QueryView& q, float* out, uint32_t* sig,
                    const AdjointOut* adj, const MisDev* mis, unsigned long long* stats) {
    if (q.count == 0) return;
    EvalArgs A = base_args(ctx, q);
    if (stats) A.stats = stats;
    set_mis(A, mis);
    A.nodes = ph.nodes;
    A.pos_r2 = ph.pos_r2;
    A.power = ph.power;
    A.inc = ph.inc;
    A.orig = ph.orig;
    A.red = ph.sel;
    A.out = out;
    A.sig = sig;
    if (adj) {
        A.grad_out = adj->grad_out;
        A.grad_media = adj->grad_media;
        A.grad_mask = (uint32_t)grad_rows(ctx.n_media) - 1u;
        A.grad_items = adj->grad_items;
    }
    const int want = ctx.tuning.photon_waves_per_block > 0 ? ctx.tuning.photon_waves_per_block
                                                           : ctx.tuning.waves_per_block;
    launch_mode<kEstPhotons>(ctx, mode, A, q, ph.n, want);
}

void launch_beams(Ctx& ctx, Mode mode, const BeamArgs& bm, const QueryView& q, float* out, uint32_t* sig,
                  const AdjointOut* adj, const MisDev* mis, unsigned long long* stats) {
    if (q.count == 0) return;
    EvalArgs A = base_args(ctx, q);
    if (stats) A.stats = stats;
    set_mis(A, mis);
    A.nodes = bm.nodes;
    A.pieces = bm.pieces;
    A.piece_flux = bm.piece_flux;
    A.orig = bm.piece_beam;
    A.end_bits = bm.end_bits;
    A.red = bm.red;
    A.out = out;
    A.sig = sig;
    if (adj) {
        A.grad_out = adj->grad_out;
        A.grad_media = adj->grad_media;
        A.grad_mask = (uint32_t)grad_rows(ctx.n_media) - 1u;
        A.grad_items = adj->grad_items;
    }
    launch_mode<kEstBeams>(ctx, mode, A, q, bm.pieces_n, ctx.tuning.waves_per_block);
}

void launch_rebase_nodes(Ctx& ctx, NodeDev* nodes, int64_t n, uint32_t node_off, uint32_t item_off) {
    if (n <= 0 || (node_off == 0 && item_off == 0)) return;
    hipLaunchKernelGGL(k_rebase_nodes, dim3(grid_for(n)), dim3(256), 0, ctx.stream, nodes, n, node_off, item_off);
    UPBP_HIP(hipGetLastError());
}

void prepare_batched(Ctx& ctx, int waves_per_block, bool planned) {
    const int wpb = std::min(std::max(waves_per_block, 1), 4);
    const int key = planned ? 4 + wpb : wpb;
    if (ctx.batched_key == key) return;
    const void* const kernels[2][2] = {{reinterpret_cast<const void*>(&k_eval_batched<kEstPhotons, false>),
                                        reinterpret_cast<const void*>(&k_eval_batched<kEstBeams, false>)},
                                       {reinterpret_cast<const void*>(&k_eval_batched<kEstPhotons, true>),
                                        reinterpret_cast<const void*>(&k_eval_batched<kEstBeams, true>)}};
    for (int e = 0; e < 2; ++e) {
        int n = 0;
        UPBP_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernels[planned][e], wpb * kWave, 0));
        ctx.batched_per_cu[e] = std::max(n, 1);
    }
    ctx.batched_key = key;
}

uint32_t batched_log_most(int64_t items) {
    uint32_t lg = 0;
    while (items >= kSplitFrom && (2u << lg) <= kPlanMost && (kSplitItems << (lg + 1)) <= items) ++lg;
    return lg;
}

static EvalArgs batched_args(Ctx& ctx, const BatchSplit& split, const MergedDev& merged, int which) {
    EvalArgs A = {};
    A.media = ctx.media.as<MediumDev>();
    A.n_media = ctx.n_media;
    A.stats = ctx.stats.as<unsigned long long>();
    A.frustum_leaf = (uint32_t)ctx.tuning.frustum_leaf;  // merged nodes keep node index == item index offsets
    if (which == kEstPhotons) {
        A.nodes = merged.ph_nodes;
        A.pos_r2 = merged.ph_pos_r2;
        A.power = merged.ph_power;
        A.inc = merged.ph_inc;
    } else {
        A.nodes = merged.bm_nodes;
        A.pieces = merged.bm_pieces;
        A.piece_flux = merged.bm_flux;
    }
    if (split.planned) {
        const TilePlan& p = split.plan[which];
        A.tasks = p.tasks;
        A.plan = p.words;
        A.rows = p.rows;
        A.shift = part_shift(kSplitFrom);  // instances are small: 64 items per block from 8 parts on
    }
    return A;
}

template <int EST>
static void plan_batched(Ctx& ctx, const InstanceDev* inst, int n_inst, int64_t tiles, const BatchSplit& split,
                         const MergedDev& merged) {
    const TilePlan& p = split.plan[EST];
    const PlanArgs P = {tiles, (uint32_t)kPlanWaves, 0, 0, false, p.cost, p.info, p.tasks, p.words};
    hipLaunchKernelGGL(k_tile_cost_batched<EST>, dim3(grid_for(tiles, 4)), dim3(256), 0, ctx.stream,
                       batched_args(ctx, split, merged, EST), P, inst, n_inst);
    launch_plan(ctx, P);
}

void launch_batched_plan(Ctx& ctx, const InstanceDev* inst, int n_inst, int64_t total_tiles, const BatchSplit& split,
                         const MergedDev& merged, int which) {
    if (!split.planned) return;
    if (which == kEstPhotons)
        plan_batched<kEstPhotons>(ctx, inst, n_inst, total_tiles, split, merged);
    else
        plan_batched<kEstBeams>(ctx, inst, n_inst, total_tiles, split, merged);
}

void launch_batched(Ctx& ctx, const InstanceDev* inst, int n_inst, int64_t total_tiles, uint32_t* counters,
                    const BatchSplit& split, const MergedDev& merged, int which, int grid_blocks, int waves_per_block) {
    const EvalArgs A = batched_args(ctx, split, merged, which);
    const int wpb = std::min(std::max(waves_per_block, 1), 4);
    if (grid_blocks <= 0) {
        // persistent grid: as many blocks as can be resident at once on every CU
        UPBP_REQUIRE(ctx.batched_key == (split.planned ? 4 + wpb : wpb) && ctx.batched_per_cu[which] > 0, UPBP_EDEVICE,
                     "batched occupancy not prepared");
        grid_blocks = ctx.num_cus * ctx.batched_per_cu[which];
    }
    const auto kernel = which == kEstPhotons
                            ? (split.planned ? k_eval_batched<kEstPhotons, true> : k_eval_batched<kEstPhotons, false>)
                            : (split.planned ? k_eval_batched<kEstBeams, true> : k_eval_batched<kEstBeams, false>);
    hipLaunchKernelGGL(kernel, dim3(grid_blocks), dim3((unsigned)(wpb * kWave)), 0, ctx.stream, A, inst, n_inst,
                       total_tiles, counters + which);
    UPBP_HIP(hipGetLastError());
    if (!split.planned) return;
    hipLaunchKernelGGL(k_sum_rows_batched, dim3(grid_for(total_tiles, 4)), dim3(256), 0, ctx.stream, inst, n_inst,
                       total_tiles, which == kEstBeams, split.plan[which].info, split.plan[which].rows);
    UPBP_HIP(hipGetLastError());
}

void launch_query_keys(Ctx& ctx, const QueryView& q, const float* lo, const float* hi, bool by_direction,
                       uint32_t* keys, uint32_t* idx) {
    float sc[3];
    for (int a = 0; a < 3; ++a) {
        const float e = hi[a] - lo[a];
        sc[a] = e > 0.f ? 1024.f / e : 0.f;
    }
    hipLaunchKernelGGL(k_query_keys, dim3(grid_for(q.count)), dim3(256), 0, ctx.stream, q.count, q.origin,
                       q.direction, q.offsets, q.segments, lo[0], lo[1], lo[2], sc[0], sc[1], sc[2],
                       by_direction, keys, idx);
    UPBP_HIP(hipGetLastError());
}

void launch_clear_u64(Ctx& ctx, uint64_t* p, int64_t n) {
    hipLaunchKernelGGL(k_clear_u64, dim3(grid_for(n)), dim3(256), 0, ctx.stream, (unsigned long long*)p, n);
    UPBP_HIP(hipGetLastError());
}

void launch_clear_f32(Ctx& ctx, float* p, int64_t n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(k_clear_f32, dim3(grid_for(n)), dim3(256), 0, ctx.stream, p, n);
    UPBP_HIP(hipGetLastError());
}

void launch_fill_u32(Ctx& ctx, uint32_t* p, uint32_t v, int64_t n) {
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n)), dim3(256), 0, ctx.stream, p, v, n);
    UPBP_HIP(hipGetLastError());
}

void launch_combine_media_grads(Ctx& ctx, const float* gm, const float* sign, int n_media, float* gs, float* ga) {
    hipLaunchKernelGGL(k_combine_media, dim3(grid_for(3 * n_media)), dim3(256), 0, ctx.stream, gm, grad_rows(n_media), sign,
                       n_media, gs, ga);
    UPBP_HIP(hipGetLastError());
}

// EmbreeBre::evalBreBruteForce (SmallUPBP/src/Bre/Bre.cxx:980-1029), the reference's debug
// estimate: one wave per query, the lanes taking every 64th kept photon; a photon inside the
// query's [min_t, max_t] disc test adds ((flux exp(-sigma_t t)) rho(d, inc)) / r^2, with the
// attenuation from the ray origin and the phase of the stored incoming direction as given
// (PhaseFunction::Evaluate(d, incDir)), and the wave's sum is scaled by sigma_s / pi.
__global__ __launch_bounds__(256) void k_bre_brute(int64_t nq, int64_t np, const float4* __restrict__ pos_r2,
                                                   const float4* __restrict__ power, const float4* __restrict__ inc,
                                                   const float* origin, const float* direction, const float* min_t,
                                                   const float* max_t, const int32_t* medium, const MediumDev* media,
                                                   int32_t n_media, float* out, uint32_t* err) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t q = (blockIdx.x * (int64_t)blockDim.x + threadIdx.x) / kWave;  // wave-uniform
    if (q >= nq) return;
    const int32_t mid = medium[q];
    if (mid < 0 || mid >= n_media) {
        if (lane == 0) {
            atomicOr(err, kErrBadMedium);
            out[3 * q] = out[3 * q + 1] = out[3 * q + 2] = 0.f;
        }
        return;
    }
    const MediumDev& M = media[mid];
    const float ox = origin[3 * q], oy = origin[3 * q + 1], oz = origin[3 * q + 2];
    const float dx = direction[3 * q], dy = direction[3 * q + 1], dz = direction[3 * q + 2];
    const float t0 = min_t[q], t1 = max_t[q];
    float a0 = 0.f, a1 = 0.f, a2 = 0.f;
    for (int64_t i = lane; i < np; i += kWave) {
        const float4 p = pos_r2[i];
        float t, sq;
        if (test_bre(ox, oy, oz, dx, dy, dz, t0, t1, p.x, p.y, p.z, p.w, t, sq)) {
            const float4 f = power[i];
            const float4 in = inc[i];
            const float rho = phase_pdf(M.g, M.isotropic != 0, -dot3(in.x, in.y, in.z, dx, dy, dz));
            a0 += ((f.x * fast_exp(-t * M.st[0])) * rho) / p.w;
            a1 += ((f.y * fast_exp(-t * M.st[1])) * rho) / p.w;
            a2 += ((f.z * fast_exp(-t * M.st[2])) * rho) / p.w;
        }
    }
    a0 = wave_sum_dpp(a0);
    a1 = wave_sum_dpp(a1);
    a2 = wave_sum_dpp(a2);
    if (lane == 0) {
        out[3 * q] = (a0 * M.ss[0]) * kInvPi;
        out[3 * q + 1] = (a1 * M.ss[1]) * kInvPi;
        out[3 * q + 2] = (a2 * M.ss[2]) * kInvPi;
    }
}

void bre_eval_brute_force(Ctx& ctx, const Bre& b, const float* origin, const float* direction, const float* min_t,
                          const float* max_t, const int32_t* medium, int64_t count, float* out) {
    if (count == 0) return;
    DevBuf err;
    err.ensure(4);
    launch_fill_u32(ctx, err.as<uint32_t>(), 0u, 1);
    const int64_t threads = count * kWave;
    hipLaunchKernelGGL(k_bre_brute, dim3(grid_for(threads)), dim3(256), 0, ctx.stream, count, b.n,
                       b.pos_r2.as<float4>(), b.power.as<float4>(), b.inc.as<float4>(), origin, direction, min_t,
                       max_t, medium, ctx.media.as<MediumDev>(), (int32_t)ctx.n_media, out, err.as<uint32_t>());
    UPBP_HIP(hipGetLastError());
    uint32_t e = 0;
    UPBP_HIP(hipMemcpyAsync(&e, err.p, 4, hipMemcpyDeviceToHost, ctx.stream));
    UPBP_HIP(hipStreamSynchronize(ctx.stream));
    UPBP_REQUIRE(!(e & kErrBadMedium), UPBP_EINVAL, "query medium outside the media table");
}

}  // namespace upbp
