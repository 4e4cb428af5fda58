// lbvh.hip -- GPU linear BVH build (Morton codes, radix sort, boxes of aligned item runs, Karras
// hierarchy emitted as 64-byte two-box nodes).
//
// Replaces the Embree BVH4 binned-SAH build over photon cubes
// (SmallUPBP/src/Bre/Bre.cxx:492-507, embree-2.0/embree/bvh4/bvh4.cpp:71) and
// the beam grid build (SmallUPBP/src/Beams/Grid.hxx:223-279). Culling only:
// node boxes are widened by a margin so that no item whose predicate accepts a
// query is ever culled; the hit set is then the brute-force hit set.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>

#include "upbp_internal.hpp"

namespace upbp {

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ uint32_t f2ord(float f) {
    uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__host__ __device__ inline float ord2f(uint32_t u) {
    uint32_t b = (u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u;
    float f;
    memcpy(&f, &b, 4);
    return f;
}

// bounds[0..2] = min item-box lo, [3..5] = max item-box hi,
// [6..8] = min centroid, [9..11] = max centroid (order-preserving uint encoding).
// Per-block partial bounds; k_bounds_final folds the partials (no global atomics:
// thousands of atomics on the same twelve words serialise).
__global__ __launch_bounds__(kBlock) void k_bounds(int64_t n, const float4* lo, const float4* hi,
                                                   uint32_t* partial) {
    uint32_t v[12];
    for (int k = 0; k < 12; ++k) v[k] = ((k / 3) % 2 == 0) ? 0xFFFFFFFFu : 0u;
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        float4 l = lo[i], h = hi[i];
        float c[3] = {0.5f * (l.x + h.x), 0.5f * (l.y + h.y), 0.5f * (l.z + h.z)};
        float ll[3] = {l.x, l.y, l.z}, hh[3] = {h.x, h.y, h.z};
        for (int a = 0; a < 3; ++a) {
            v[a] = min(v[a], f2ord(ll[a]));
            v[3 + a] = max(v[3 + a], f2ord(hh[a]));
            v[6 + a] = min(v[6 + a], f2ord(c[a]));
            v[9 + a] = max(v[9 + a], f2ord(c[a]));
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        for (int k = 0; k < 12; ++k) {
            uint32_t o = __shfl_xor(v[k], off, 64);
            v[k] = ((k / 3) % 2 == 0) ? min(v[k], o) : max(v[k], o);
        }
    }
    __shared__ uint32_t sh[kBlock / 64][12];
    const int w = threadIdx.x / 64;
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 12; ++k) sh[w][k] = v[k];
    __syncthreads();
    if (threadIdx.x < 12) {
        const int k = threadIdx.x;
        uint32_t r = sh[0][k];
        for (int j = 1; j < (int)(blockDim.x / 64); ++j) r = ((k / 3) % 2 == 0) ? min(r, sh[j][k]) : max(r, sh[j][k]);
        partial[(size_t)blockIdx.x * 12 + k] = r;
    }
}

// One wave per bound component: its lanes stride over the per-block partials, then a wave
// reduction (a single thread per component took ~125 us over 1024 partials).
__global__ void k_bounds_final(int nb, const uint32_t* partial, uint32_t* b) {
    const int k = threadIdx.x / 64, lane = threadIdx.x & 63;
    if (k >= 12) return;  // whole waves
    const bool is_min = (k / 3) % 2 == 0;
    uint32_t r = is_min ? 0xFFFFFFFFu : 0u;
    for (int i = lane; i < nb; i += 64) {
        const uint32_t v = partial[(size_t)i * 12 + k];
        r = is_min ? min(r, v) : max(r, v);
    }
    for (int off = 32; off > 0; off >>= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)r, off, 64);
        r = is_min ? min(r, o) : max(r, o);
    }
    if (lane == 0) b[k] = r;
}

__device__ __forceinline__ uint64_t spread21(uint64_t x) {
    x &= 0x1fffffull;
    x = (x | (x << 32)) & 0x1f00000000ffffull;
    x = (x | (x << 16)) & 0x1f0000ff0000ffull;
    x = (x | (x << 8)) & 0x100f00f00f00f00full;
    x = (x | (x << 4)) & 0x10c30c30c30c30c3ull;
    x = (x | (x << 2)) & 0x1249249249249249ull;
    return x;
}

__global__ __launch_bounds__(kBlock) void k_morton(int64_t n, const float4* lo, const float4* hi,
                                                   const uint32_t* b, uint64_t* keys, uint32_t* vals) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n) return;
    float4 l = lo[i], h = hi[i];
    float c[3] = {0.5f * (l.x + h.x), 0.5f * (l.y + h.y), 0.5f * (l.z + h.z)};
    uint64_t q[3];
    for (int a = 0; a < 3; ++a) {
        float mn = ord2f(b[6 + a]), mx = ord2f(b[9 + a]);
        float ext = mx - mn;
        float u = ext > 0.f ? (c[a] - mn) / ext : 0.5f;
        u = fminf(fmaxf(u, 0.f), 1.f);
        q[a] = (uint64_t)(u * 2097151.0f);
    }
    keys[i] = (spread21(q[0]) << 2) | (spread21(q[1]) << 1) | spread21(q[2]);
    vals[i] = (uint32_t)i;
}

// Length of the common prefix of keys i and j (index-tie-broken), -1 out of range.
__device__ __forceinline__ int delta(const uint64_t* keys, int64_t n, int64_t i, int64_t j) {
    if (j < 0 || j >= n) return -1;
    uint64_t a = keys[i], b = keys[j];
    if (a == b) return 64 + __clz((uint32_t)(i ^ j));
    return __clzll(a ^ b);
}

// ---- boxes of item ranges ------------------------------------------------------
// A node's box is the box of a run of sorted items. Instead of refitting the tree bottom-up (which took a
// parent walk, a sort of the nodes by depth and a launch per level), the boxes of aligned runs of 16,
// 256, 4096, ... items are kept, and any run's box is put together from at most 30 of them per level:
// min and max are exact, so the boxes are the refit's. Every node is then independent of the others:
// three to six launches instead of about 45, no wait for the host in between, and the items are read in
// sorted order once instead of through the permutation at every leaf. Bound by launches at small counts
// and by the reads of keys and boxes at large ones. Building photons and beams of 150k paths with
// radii from neighbours (five trees): 4890 us with the refit, 3930 us so.
constexpr int kRun = 16;
constexpr int kBoxLevels = 9;  // runs of 16^0 .. 16^8 items: more than 2^31

struct BoxLevels {
    const float4* lo[kBoxLevels];
    const float4* hi[kBoxLevels];
};

__device__ __forceinline__ void box_merge(float4& lo, float4& hi, const float4& l, const float4& h) {
    lo = make_float4(fminf(lo.x, l.x), fminf(lo.y, l.y), fminf(lo.z, l.z), 0.f);
    hi = make_float4(fmaxf(hi.x, h.x), fmaxf(hi.y, h.y), fmaxf(hi.z, h.z), 0.f);
}

// The boxes of runs of 16 and of 256 of n boxes (one block of 256 threads per run of 256), which are
// first brought into sorted order where order is given (then written to lo0 / hi0 too).
__global__ __launch_bounds__(kBlock) void k_box_runs(int64_t n, const uint32_t* __restrict__ order,
                                                     const float4* __restrict__ lo, const float4* __restrict__ hi,
                                                     float4* __restrict__ lo0, float4* __restrict__ hi0,
                                                     float4* __restrict__ lo1, float4* __restrict__ hi1,
                                                     float4* __restrict__ lo2, float4* __restrict__ hi2) {
    static_assert(kBlock == kRun * kRun, "one block per run of runs");
    __shared__ float4 sl[kRun], sh[kRun];
    const int64_t i = blockIdx.x * (int64_t)kBlock + threadIdx.x;
    float4 l = make_float4(INFINITY, INFINITY, INFINITY, 0.f), h = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
    if (i < n) {
        const int64_t k = order ? (int64_t)order[i] : i;
        l = lo[k];
        h = hi[k];
        if (order) {
            lo0[i] = l;
            hi0[i] = h;
        }
    }
    for (int pass = 0; pass < 2; ++pass) {
        for (int off = 1; off < kRun; off <<= 1)
            box_merge(l, h,
                      make_float4(__shfl_xor(l.x, off, kRun), __shfl_xor(l.y, off, kRun), __shfl_xor(l.z, off, kRun), 0.f),
                      make_float4(__shfl_xor(h.x, off, kRun), __shfl_xor(h.y, off, kRun), __shfl_xor(h.z, off, kRun), 0.f));
        if (pass == 1) {
            if (threadIdx.x == 0) {
                lo2[blockIdx.x] = l;
                hi2[blockIdx.x] = h;
            }
            return;
        }
        if (threadIdx.x % kRun == 0) {
            sl[threadIdx.x / kRun] = l;
            sh[threadIdx.x / kRun] = h;
            if (i < n) {
                lo1[i / kRun] = l;
                hi1[i / kRun] = h;
            }
        }
        __syncthreads();
        l = sl[threadIdx.x % kRun];
        h = sh[threadIdx.x % kRun];
    }
}

// The box of the sorted items [a, b).
__device__ __forceinline__ void box_of(const BoxLevels& L, uint32_t a, uint32_t b, float4& lo, float4& hi) {
    lo = make_float4(INFINITY, INFINITY, INFINITY, 0.f);
    hi = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.f);
#pragma unroll 1
    for (int t = 0; a < b; ++t, a /= kRun, b /= kRun) {
        const float4 *l = L.lo[t], *h = L.hi[t];
        for (; a < b && a % kRun != 0; ++a) box_merge(lo, hi, l[a], h[a]);
        for (; a < b && b % kRun != 0; --b) box_merge(lo, hi, l[b - 1], h[b - 1]);
    }
}

// Margin that keeps the float slab test conservative for every accepted item.
__host__ __device__ inline float box_margin(const float lo[3], const float hi[3]) {
    float m = 1e-3f;
    for (int a = 0; a < 3; ++a) m = fmaxf(m, fmaxf(fmaxf(fabsf(lo[a]), fabsf(hi[a])), hi[a] - lo[a]));
    return 1e-5f * m;
}

// Karras (HPG 2012) binary radix tree, emitted as two-box nodes: internal node i in [0, n-2] of the
// sorted keys with its children's boxes. A child of at most leaf_size items becomes a leaf.
__global__ __launch_bounds__(kBlock) void k_nodes(int64_t n, const uint64_t* __restrict__ keys, int leaf_size,
                                                  const uint32_t* __restrict__ bounds, BoxLevels L,
                                                  NodeDev* __restrict__ nodes) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = delta(keys, n, i, i - d);
    int64_t lmax = 2;
    while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int64_t l = 0;
    for (int64_t t = lmax >> 1; t >= 1; t >>= 1)
        if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
    const int64_t j = i + l * d;
    const int dnode = delta(keys, n, i, j);
    int64_t s = 0;
    int64_t t = l;
    do {
        t = (t + 1) >> 1;
        if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    const int64_t gamma = i + s * d + (d < 0 ? -1 : 0);
    const int64_t first = i < j ? i : j, last = i < j ? j : i;
    // children: the items [first, gamma] and [gamma + 1, last]; an inner child is node gamma or gamma + 1
    float lo[3], hi[3];
    for (int a = 0; a < 3; ++a) {
        lo[a] = ord2f(bounds[a]);
        hi[a] = ord2f(bounds[3 + a]);
    }
    const float eps = box_margin(lo, hi);
    uint32_t ref[2], cnt[2];
    float4 bl[2], bh[2];
    for (int c = 0; c < 2; ++c) {
        const uint32_t from = (uint32_t)(c == 0 ? first : gamma + 1), to = (uint32_t)(c == 0 ? gamma : last);
        const uint32_t child = (uint32_t)(c == 0 ? gamma : gamma + 1), count = to - from + 1u;
        box_of(L, from, to + 1u, bl[c], bh[c]);
        if ((int64_t)count <= leaf_size || count == 1u) {
            ref[c] = from;
            cnt[c] = count;
        } else {
            // the subtree's size and where its items start, for traversals that take a
            // small subtree as one leaf
            ref[c] = child;
            cnt[c] = kInner | (from == child ? 0u : kSpanEnds) | min(count, kSpanMask - 1u);
        }
        bl[c] = make_float4(bl[c].x - eps, bl[c].y - eps, bl[c].z - eps, 0.f);
        bh[c] = make_float4(bh[c].x + eps, bh[c].y + eps, bh[c].z + eps, 0.f);
    }
    NodeDev nd;
    nd.a = make_float4(bl[0].x, bl[0].y, bl[0].z, bh[0].x);
    nd.b = make_float4(bh[0].y, bh[0].z, bl[1].x, bl[1].y);
    nd.c = make_float4(bl[1].z, bh[1].x, bh[1].y, bh[1].z);
    nd.r = make_uint4(ref[0], ref[1], cnt[0], cnt[1]);
    nodes[i] = nd;
}

__global__ void k_iota(int64_t n, uint32_t* v) {
    int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i < n) v[i] = (uint32_t)i;
}

inline unsigned grid_for(int64_t n, int block = kBlock) {
    int64_t g = (n + block - 1) / block;
    return (unsigned)std::max<int64_t>(1, g);
}

}  // namespace

void sort_pairs_u64(Ctx& ctx, uint64_t* keys_in, uint64_t* keys_out, uint32_t* vals_in,
                    uint32_t* vals_out, int64_t n, int end_bit) {
    size_t bytes = 0;
    UPBP_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, keys_in, keys_out, vals_in, vals_out,
                                                (int)n, 0, end_bit, ctx.stream));
    ctx.sort_tmp.ensure(bytes);
    UPBP_HIP(hipcub::DeviceRadixSort::SortPairs(ctx.sort_tmp.p, bytes, keys_in, keys_out, vals_in,
                                                vals_out, (int)n, 0, end_bit, ctx.stream));
}

void sort_pairs_u32(Ctx& ctx, uint32_t* keys_in, uint32_t* keys_out, uint32_t* vals_in,
                    uint32_t* vals_out, int64_t n, int end_bit) {
    size_t bytes = 0;
    UPBP_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, keys_in, keys_out, vals_in, vals_out,
                                                (int)n, 0, end_bit, ctx.stream));
    ctx.sort_tmp.ensure(bytes);
    UPBP_HIP(hipcub::DeviceRadixSort::SortPairs(ctx.sort_tmp.p, bytes, keys_in, keys_out, vals_in,
                                                vals_out, (int)n, 0, end_bit, ctx.stream));
}

size_t sort_pairs_u32_temp_bytes(int64_t n, int end_bit) {
    size_t bytes = 0;
    UPBP_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (uint32_t*)nullptr, (uint32_t*)nullptr,
                                                (uint32_t*)nullptr, (uint32_t*)nullptr, (int)n, 0, end_bit,
                                                (hipStream_t)0));
    return bytes;
}

void sort_pairs_u32_in(Ctx& ctx, void* tmp, size_t tmp_bytes, uint32_t* keys_in, uint32_t* keys_out,
                       uint32_t* vals_in, uint32_t* vals_out, int64_t n, int end_bit) {
    size_t bytes = 0;
    UPBP_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, keys_in, keys_out, vals_in, vals_out,
                                                (int)n, 0, end_bit, ctx.stream));
    UPBP_REQUIRE(bytes <= tmp_bytes, UPBP_EDEVICE, "radix sort needs more temporary storage than the workspace holds");
    UPBP_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, bytes, keys_in, keys_out, vals_in, vals_out, (int)n, 0,
                                                end_bit, ctx.stream));
}

void exclusive_scan_u32(Ctx& ctx, const uint32_t* in, uint32_t* out, int64_t n) {
    size_t bytes = 0;
    UPBP_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, (int)n, ctx.stream));
    ctx.sort_tmp.ensure(bytes);
    UPBP_HIP(hipcub::DeviceScan::ExclusiveSum(ctx.sort_tmp.p, bytes, in, out, (int)n, ctx.stream));
}

void build_lbvh(Ctx& ctx, int64_t n, const float4* box_lo, const float4* box_hi, int leaf_size,
                Lbvh& out, DevBuf& out_order) {
    UPBP_REQUIRE(n > 0 && n < (int64_t)0x7FFFFFFF, UPBP_EINVAL, "LBVH item count out of range");
    hipStream_t st = ctx.stream;
    out.n_items = n;
    TmpBuf bounds(ctx.tmp), partial(ctx.tmp);
    bounds.ensure(12 * 4);
    const unsigned gb = std::min<unsigned>(grid_for(n), 1024u);
    partial.ensure((size_t)gb * 12 * 4);
    hipLaunchKernelGGL(k_bounds, dim3(gb), dim3(kBlock), 0, st, n, box_lo, box_hi, partial.as<uint32_t>());
    UPBP_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_bounds_final, dim3(1), dim3(12 * 64), 0, st, (int)gb, partial.as<uint32_t>(),
                       bounds.as<uint32_t>());
    UPBP_HIP(hipGetLastError());
    // waits for everything queued so far and takes the item bounds
    const auto take_bounds = [&] {
        uint32_t hb[12];
        UPBP_HIP(hipMemcpyAsync(hb, bounds.p, sizeof(hb), hipMemcpyDeviceToHost, st));
        UPBP_HIP(hipStreamSynchronize(st));
        for (int a = 0; a < 3; ++a) {
            out.lo[a] = ord2f(hb[a]);
            out.hi[a] = ord2f(hb[3 + a]);
            UPBP_REQUIRE(std::isfinite(out.lo[a]) && std::isfinite(out.hi[a]), UPBP_ENONFINITE,
                         "non-finite item bounds");
        }
    };
    out_order.ensure((size_t)n * 4);
    if (n <= leaf_size) {
        // one node: child 0 is a leaf with every item, child 1 absent
        take_bounds();
        const float eps = box_margin(out.lo, out.hi);
        hipLaunchKernelGGL(k_iota, dim3(grid_for(n)), dim3(kBlock), 0, st, n, out_order.as<uint32_t>());
        NodeDev nd;
        nd.a = make_float4(out.lo[0] - eps, out.lo[1] - eps, out.lo[2] - eps, out.hi[0] + eps);
        nd.b = make_float4(out.hi[1] + eps, out.hi[2] + eps, 0.f, 0.f);
        nd.c = make_float4(0.f, 0.f, 0.f, 0.f);
        nd.r = make_uint4(0u, 0u, (uint32_t)n, kInvalid);
        out.nodes.ensure(sizeof(NodeDev));
        UPBP_HIP(hipMemcpyAsync(out.nodes.p, &nd, sizeof(nd), hipMemcpyHostToDevice, st));
        out.n_nodes = 1;
        UPBP_HIP(hipStreamSynchronize(st));
        return;
    }
    TmpBuf keys(ctx.tmp), keys2(ctx.tmp), vals(ctx.tmp);
    keys.ensure((size_t)n * 8);
    keys2.ensure((size_t)n * 8);
    vals.ensure((size_t)n * 4);
    hipLaunchKernelGGL(k_morton, dim3(grid_for(n)), dim3(kBlock), 0, st, n, box_lo, box_hi,
                       bounds.as<uint32_t>(), keys.as<uint64_t>(), vals.as<uint32_t>());
    UPBP_HIP(hipGetLastError());
    sort_pairs_u64(ctx, keys.as<uint64_t>(), keys2.as<uint64_t>(), vals.as<uint32_t>(),
                   out_order.as<uint32_t>(), n, 63);
    // boxes of aligned runs: level t holds ceil(n / 16^t) of them, two levels per launch
    int64_t count[kBoxLevels], at[kBoxLevels], total = 0;
    for (int t = 0; t < kBoxLevels; ++t) {
        count[t] = t == 0 ? n : (count[t - 1] + kRun - 1) / kRun;
        at[t] = total;
        total += count[t];
    }
    TmpBuf run_lo(ctx.tmp), run_hi(ctx.tmp);
    run_lo.ensure((size_t)total * 16);
    run_hi.ensure((size_t)total * 16);
    BoxLevels L;
    for (int t = 0; t < kBoxLevels; ++t) {
        L.lo[t] = run_lo.as<float4>() + at[t];
        L.hi[t] = run_hi.as<float4>() + at[t];
    }
    for (int t = 0; t + 2 < kBoxLevels && (t == 0 || count[t] > 1); t += 2) {
        float4 *lo = run_lo.as<float4>(), *hi = run_hi.as<float4>();
        hipLaunchKernelGGL(k_box_runs, dim3((unsigned)count[t + 2]), dim3(kBlock), 0, st, count[t],
                           t == 0 ? out_order.as<uint32_t>() : (const uint32_t*)nullptr, t == 0 ? box_lo : lo + at[t],
                           t == 0 ? box_hi : hi + at[t], lo + at[0], hi + at[0], lo + at[t + 1], hi + at[t + 1],
                           lo + at[t + 2], hi + at[t + 2]);
        UPBP_HIP(hipGetLastError());
    }
    out.nodes.ensure((size_t)(n - 1) * sizeof(NodeDev));
    out.n_nodes = n - 1;
    hipLaunchKernelGGL(k_nodes, dim3(grid_for(n - 1)), dim3(kBlock), 0, st, n, keys2.as<uint64_t>(), leaf_size,
                       bounds.as<uint32_t>(), L, out.nodes.as<NodeDev>());
    UPBP_HIP(hipGetLastError());
    take_bounds();
}

}  // namespace upbp
