// morton.hip -- SpatialAccel::build: 30-bit Morton codes on a scene box,
// their stable sort, and the linear BVH over the sorted codes.
//
// Replaces core/src/spatial_accel.cu: codes 11-40, host inverse extent
// 139-148, sort on bits [0,30) 158-179, Karras internal nodes 44-100, leaf
// boxes 102-113 (radius 0, as build() uses).  The internal boxes, which the
// reference leaves for later, are filled here as well.
#include <algorithm>

#include "radix_sort.hpp"
#include "wsim_internal.hpp"

namespace wsim {
namespace {

// Bit b of a 10-bit value moves to bit 3b.
__device__ inline u32 spread10(u32 v) {
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// Quantise one normalised coordinate to [0, 1023] (spatial_accel.cu:21-26).
__device__ inline u32 quant10(float p, float lo, float inv) {
    const float t = (p - lo) * inv;
    return static_cast<u32>(fminf(fmaxf(t * 1024.0f, 0.0f), 1023.0f));
}

// Codes and original indices; workgroup t writes the sort's tile t and counts
// the first digit of its codes (radix_count_*).
__global__ __launch_bounds__(kRadixThreads) void k_morton(const float* __restrict__ xyz, u32 n,
                                                          float mx, float my, float mz, float ix,
                                                          float iy, float iz,
                                                          u32* __restrict__ codes,
                                                          u32* __restrict__ vals, u32 dmask,
                                                          u32* __restrict__ hist, u32 tiles) {
    __shared__ u32 cnt[256];
    radix_count_begin(cnt);
#pragma unroll
    for (int r = 0; r < kRadixTile / kRadixThreads; ++r) {
        const u32 i = blockIdx.x * kRadixTile + r * kRadixThreads + threadIdx.x;
        if (i >= n) continue;
        const u64 o = 3ull * i;
        const u32 qx = quant10(xyz[o], mx, ix);
        const u32 qy = quant10(xyz[o + 1], my, iy);
        const u32 qz = quant10(xyz[o + 2], mz, iz);
        const u32 code = (spread10(qx) << 2) | (spread10(qy) << 1) | spread10(qz);
        codes[i] = code;
        vals[i] = i;
        radix_count_key(cnt, code & dmask);
    }
    radix_count_end(cnt, dmask, hist, tiles);
}

__device__ __forceinline__ void box_union(float* c, const float* a, const float* b) {
    for (int k = 0; k < 3; ++k) {
        c[k] = fminf(a[k], b[k]);
        c[k + 3] = fmaxf(a[k + 3], b[k + 3]);
    }
}

// Internal boxes without inter-thread ordering: a segment tree over the
// sorted leaves (node t of level k unions the leaves [t 2^k, (t + 1) 2^k)),
// then every internal node unions the O(log n) segment-tree boxes that tile
// its leaf range.  min and max are exact, so the result equals the bottom-up
// union of the children.
constexpr int kSegThreads = 512;
constexpr int kSegNodes = 2 * kSegThreads;  // nodes of the lowest level per workgroup
constexpr int kSegLevels = 10;              // levels one launch adds above it
static_assert(kSegNodes == 1 << kSegLevels, "a workgroup's subtree ends in one node");
constexpr int kMaxLevels = 33;
struct SegTree {
    float* level[kMaxLevels];  // level 0: the leaf boxes
    u32 m[kMaxLevels];         // nodes per level
    int levels;
};

// The subtrees of kSegNodes nodes of level `base`, a workgroup each: ten
// levels per launch in LDS, every level written once, instead of one launch a
// level (a million leaves: 20 launches of 2.4 us and their gaps before, two
// launches now).  LEAF: level 0 is gathered from the points (radius 0, as
// spatial_accel.cu:102-113) and written too.
template <bool LEAF>
__global__ __launch_bounds__(kSegThreads) void k_seg_levels(const float* __restrict__ xyz,
                                                            const u32* __restrict__ sorted,
                                                            SegTree T, int base) {
    __shared__ float s[6][kSegNodes];
    const u32 first = blockIdx.x * kSegNodes;
    const u32 cnt = min(T.m[base] - first, static_cast<u32>(kSegNodes));
    float* const low = T.level[base] + 6ull * first;
    if constexpr (LEAF) {
        for (u32 i = threadIdx.x; i < cnt; i += kSegThreads) {
            const u64 o = 3ull * sorted[first + i];
#pragma unroll
            for (int k = 0; k < 3; ++k) s[k][i] = s[k + 3][i] = xyz[o + k];
        }
        __syncthreads();
        for (u32 f = threadIdx.x; f < 6 * cnt; f += kSegThreads) low[f] = s[f % 6][f / 6];
    } else {
        for (u32 f = threadIdx.x; f < 6 * cnt; f += kSegThreads) s[f % 6][f / 6] = low[f];
        __syncthreads();
    }
    u32 below = cnt;
    for (int j = 1; j <= kSegLevels && base + j < T.levels; ++j) {
        const u32 m = (below + 1) / 2;
        const u32 t = threadIdx.x;
        float c[6];
        if (t < m) {
#pragma unroll
            for (int k = 0; k < 6; ++k) c[k] = s[k][2 * t];
            if (2 * t + 1 < below) {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    c[k] = fminf(c[k], s[k][2 * t + 1]);
                    c[k + 3] = fmaxf(c[k + 3], s[k + 3][2 * t + 1]);
                }
            }
        }
        __syncthreads();
        if (t < m) {
#pragma unroll
            for (int k = 0; k < 6; ++k) s[k][t] = c[k];
        }
        __syncthreads();
        float* const out = T.level[base + j] + 6ull * (first >> j);
        for (u32 f = threadIdx.x; f < 6 * m; f += kSegThreads) out[f] = s[f % 6][f / 6];
        below = m;
    }
}

// Length of the common prefix of sorted leaves i and j in the total order
// (code, index): equal codes compare their indices, so every prefix is
// unique (Karras 2012; spatial_accel.cu:44-55).  -1 for j outside [0, n).
// Codes near the workgroup's nodes come from LDS.
constexpr int kKarrasThreads = 256;
constexpr int kKarrasReach = 256;  // codes kept on either side
constexpr int kKarrasWindow = kKarrasThreads + 2 * kKarrasReach;
template <class I>
struct CodeWindow {
    const u32* codes;
    const u32* window;
    I n, first;  // first: leaf of window[0]
    __device__ __forceinline__ u32 code(I j) const {
        const I k = j - first;
        return k >= 0 && k < kKarrasWindow ? window[k] : codes[j];
    }
    __device__ __forceinline__ int prefix(I i, u32 a, I j) const {
        if (j < 0 || j >= n) return -1;
        const u32 b = code(j);
        if (a == b) return 32 + __clz(static_cast<u32>(i ^ j));
        return __clz(a ^ b);
    }
};

// Internal node i of the binary radix tree over n sorted codes (Karras 2012,
// as spatial_accel.cu:57-100): the direction of its range, the range's far
// end by exponential then binary search, the split by binary search; then its
// box.  Children >= n - 1 are leaves (n - 1 + leaf index); the root's parent
// is ~0u.  Every search step waits for one code; most ranges are short, so
// the workgroup keeps the codes around its nodes in LDS (a million leaves:
// 43 us; node search 31.6 and boxes 24.6 us as two kernels reading global
// memory).  The whole build went from 242 to 182 us.
// I: index type, 32 bits while n + the search's overshoot fit.
template <class I>
__global__ __launch_bounds__(kKarrasThreads) void k_karras(const u32* __restrict__ codes, u32 n,
                                                           u32* __restrict__ left,
                                                           u32* __restrict__ right,
                                                           u32* __restrict__ parent, SegTree T,
                                                           float* __restrict__ boxes) {
    __shared__ u32 s_code[kKarrasWindow];
    const I nn = static_cast<I>(n), ni = nn - 1;
    const I block0 = static_cast<I>(blockIdx.x) * kKarrasThreads;
    const CodeWindow<I> W{codes, s_code, nn, block0 - kKarrasReach};
    for (int k = threadIdx.x; k < kKarrasWindow; k += kKarrasThreads) {
        const I j = W.first + k;
        s_code[k] = j >= 0 && j < nn ? codes[j] : 0u;
    }
    __syncthreads();
    const I i = block0 + static_cast<I>(threadIdx.x);
    if (i >= ni) return;
    if (i == 0) parent[0] = ~0u;
    const u32 ci = W.code(i);
    const I d = W.prefix(i, ci, i + 1) - W.prefix(i, ci, i - 1) > 0 ? 1 : -1;
    const int dmin = W.prefix(i, ci, i - d);
    I lmax = 2;
    while (W.prefix(i, ci, i + lmax * d) > dmin) lmax *= 2;
    I l = 0;
    for (I t = lmax / 2; t > 0; t /= 2)
        if (W.prefix(i, ci, i + (l + t) * d) > dmin) l += t;
    const I j = i + l * d;
    const int dnode = W.prefix(i, ci, j);
    I s = 0;
    for (I t = (l + 1) / 2; t > 0; t = (t == 1) ? 0 : (t + 1) / 2)
        if (W.prefix(i, ci, i + (s + t) * d) > dnode) s += t;
    const I gamma = i + s * d + (d < 0 ? -1 : 0);
    const I lo = i < j ? i : j, hi = i < j ? j : i;
    const u32 a = static_cast<u32>(lo == gamma ? ni + gamma : gamma);
    const u32 b = static_cast<u32>(hi == gamma + 1 ? ni + gamma + 1 : gamma + 1);
    left[i] = a;
    right[i] = b;
    parent[a] = static_cast<u32>(i);
    parent[b] = static_cast<u32>(i);
    // the box: segment-tree nodes that tile leaves [lo, hi]
    float acc[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    u32 el = static_cast<u32>(lo), er = static_cast<u32>(hi) + 1u;
    for (int k = 0; el < er; ++k, el >>= 1, er >>= 1) {
        const float* lev = T.level[k];
        if (el & 1u) box_union(acc, acc, lev + 6ull * el++);
        if (er & 1u) box_union(acc, acc, lev + 6ull * --er);
    }
    float* c = boxes + 6ull * static_cast<u64>(i);
    for (int k = 0; k < 6; ++k) c[k] = acc[k];
}

}  // namespace

void SpatialAccel::build(const float* positions_xyz, size_t count, const float bmin[3],
                         const float bmax[3], hipStream_t stream) {
    leaf_count_ = count;
    if (count == 0) return;
    if (count > 0xFFFFF000ull) fail(kInvalidArgument, "SpatialAccel: too many particles");
    k_[0].ensure(count);
    k_[1].ensure(count);
    v_[0].ensure(count);
    v_[1].ensure(count);
    hist_.ensure(radix_hist_elems(count));
    float inv[3];
    for (int a = 0; a < 3; ++a) {
        const float e = bmax[a] - bmin[a];
        inv[a] = e > 0 ? 1.0f / e : 0.0f;  // spatial_accel.cu:144-148
    }
    const u32 n = static_cast<u32>(count);
    const u32 tiles = radix_tiles(n);
    constexpr int kCodeBits = 30;
    k_morton<<<tiles, kRadixThreads, 0, stream>>>(positions_xyz, n, bmin[0], bmin[1], bmin[2],
                                                  inv[0], inv[1], inv[2], k_[0].data(),
                                                  v_[0].data(), radix_first_digit_mask(kCodeBits),
                                                  hist_.data(), tiles);
    WSIM_LAUNCH_CHECK();
    cur_ = radix_sort_pairs(k_[0].data(), v_[0].data(), k_[1].data(), v_[1].data(), count,
                            kCodeBits, hist_.data(), stream, true);
    boxes_.ensure(6 * (2 * count - 1));
    parent_.ensure(2 * count - 1);
    // segment tree: level 0 is the leaf part of boxes_, the others lie in seg_
    SegTree T{};
    T.m[0] = n;
    T.levels = 1;
    u64 above = 0;
    while (T.m[T.levels - 1] > 1) {
        T.m[T.levels] = (T.m[T.levels - 1] - 1u) / 2u + 1u;
        above += T.m[T.levels];
        ++T.levels;
    }
    seg_.ensure(6 * std::max<u64>(above, 1));
    T.level[0] = boxes_.data() + 6ull * (n - 1);
    u64 at = 0;
    for (int k = 1; k < T.levels; ++k) {
        T.level[k] = seg_.data() + 6ull * at;
        at += T.m[k];
    }
    k_seg_levels<true><<<div_up(n, kSegNodes), kSegThreads, 0, stream>>>(
        positions_xyz, v_[cur_].data(), T, 0);
    WSIM_LAUNCH_CHECK();
    if (count == 1) {
        WSIM_HIP(hipMemsetAsync(parent_.data(), 0xFF, sizeof(u32), stream));
        return;
    }
    for (int base = kSegLevels; base + 1 < T.levels; base += kSegLevels) {
        k_seg_levels<false><<<div_up(T.m[base], kSegNodes), kSegThreads, 0, stream>>>(
            nullptr, nullptr, T, base);
        WSIM_LAUNCH_CHECK();
    }
    left_.ensure(count - 1);
    right_.ensure(count - 1);
    const u32 nblk = div_up(n - 1, kKarrasThreads);
    if (n < (1u << 29))
        k_karras<int><<<nblk, kKarrasThreads, 0, stream>>>(k_[cur_].data(), n, left_.data(),
                                                           right_.data(), parent_.data(), T,
                                                           boxes_.data());
    else
        k_karras<long long><<<nblk, kKarrasThreads, 0, stream>>>(k_[cur_].data(), n, left_.data(),
                                                                 right_.data(), parent_.data(), T,
                                                                 boxes_.data());
    WSIM_LAUNCH_CHECK();
    // the nodes and boxes are complete for every stream when this returns
    WSIM_HIP(hipStreamSynchronize(stream));
}

}  // namespace wsim
