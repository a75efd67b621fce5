// surface.hip -- fluid surface mesh from particle positions on the GPU.
//
// Replaces the splat method of tools/particles_to_mesh.py
// (reconstruct_splat, :77-138 with load_frame :46-58), the consumer of the
// frame format downstream of sim_cli:
//   1. bounds of the points (optionally with y and z swapped, the
//      reference's sim Y-up -> Blender Z-up), padded by 4 r;
//   2. splat: +1 in the voxel (p - lo) / extent * res, truncated and
//      clipped, res = max(ceil(extent / (factor r)), 8) per axis;
//   3. Gaussian blur of the voxel counts, the three 1-D passes of
//      scipy.ndimage.gaussian_filter (truncate 4, mode 'reflect', binary64
//      sums in its order for symmetric weights, binary32 between passes);
//   4. iso = max * iso_factor in binary32 (numpy 2 scalar rules);
//   5. marching cubes with shared vertices: one vertex per grid edge whose
//      end values straddle the iso level (linear interpolation), triangles
//      from a table built from the cube faces (mc_table).
// Before the bounds, the reference's k-nearest-neighbour position smoothing
// (smooth_positions_knn :61-74) runs smooth_pre_iters times; after marching
// cubes, smooth_post_iters passes of the Laplacian mesh smoothing it asks of
// Open3D (:138-139, filter_smooth_laplacian, lambda 0.5).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "device_math.hpp"
#include "radix_sort.hpp"
#include "wsim_internal.hpp"

namespace wsim {
namespace {

constexpr int kMeshThreads = 256;
constexpr int kMaxTri = 8;  // triangles per cube configuration (the table has at most 5)

// ---- marching-cubes table ---------------------------------------------------
// Corner c of a cube sits at offset (c & 1, c >> 1 & 1, c >> 2 & 1) along the
// grid axes (0, 1, 2).  Edge a * 4 + b runs along axis a from the corner
// with bit a clear; b holds that corner's other two bits (lower axis first).
// A corner is inside when its value exceeds the iso level.  On every face,
// each run of consecutive inside corners (going round the face; diagonal
// inside corners are separate runs) is bounded by two crossing edges, which
// a surface segment joins.  The segments close into loops around the
// edge-connected inside corners, and each loop becomes a triangle fan.
// Neighbouring cubes build the same segments on their shared face, so the
// surface is closed; segments are oriented so that triangle normals point
// from the inside corners outwards.
struct McTable {
    uint8_t ntri[256];
    uint8_t tri[256][kMaxTri * 3];
};

int edge_between(int c0, int c1) {
    const int a = __builtin_ctz(static_cast<unsigned>(c0 ^ c1));
    const int base = c0 & ~(1 << a);
    int b = 0, k = 0;
    for (int ax = 0; ax < 3; ++ax) {
        if (ax == a) continue;
        b |= ((base >> ax) & 1) << k;
        ++k;
    }
    return a * 4 + b;
}

McTable build_mc_table() {
    McTable t{};
    for (int cfg = 0; cfg < 256; ++cfg) {
        auto inside = [&](int c) { return ((cfg >> c) & 1) != 0; };
        int next[12];
        for (int& e : next) e = -1;
        for (int a = 0; a < 3; ++a) {
            const int u = (a + 1) % 3, v = (a + 2) % 3;  // (u, v, a) right-handed
            for (int s = 0; s < 2; ++s) {
                int cyc[4];
                const int du[4] = {0, 1, 1, 0}, dv[4] = {0, 0, 1, 1};
                for (int m = 0; m < 4; ++m) cyc[m] = (s << a) | (du[m] << u) | (dv[m] << v);
                if (s == 0) std::swap(cyc[1], cyc[3]);  // counter-clockwise seen from outside
                for (int m = 0; m < 4; ++m) {
                    if (!inside(cyc[m]) || inside(cyc[(m + 3) % 4])) continue;  // run start
                    int k = m;
                    while (inside(cyc[(k + 1) % 4])) k = (k + 1) % 4;
                    const int e_in = edge_between(cyc[(m + 3) % 4], cyc[m]);
                    const int e_out = edge_between(cyc[k], cyc[(k + 1) % 4]);
                    next[e_in] = e_out;
                }
            }
        }
        bool seen[12] = {};
        int nt = 0;
        for (int e0 = 0; e0 < 12; ++e0) {
            if (next[e0] < 0 || seen[e0]) continue;
            int loop[12], len = 0;
            for (int e = e0; !seen[e]; e = next[e]) {
                seen[e] = true;
                loop[len++] = e;
            }
            for (int k = 1; k + 1 < len; ++k) {
                if (nt >= kMaxTri) fail(kRuntimeError, "marching-cubes table overflow");
                t.tri[cfg][3 * nt + 0] = static_cast<uint8_t>(loop[0]);
                t.tri[cfg][3 * nt + 1] = static_cast<uint8_t>(loop[k]);
                t.tri[cfg][3 * nt + 2] = static_cast<uint8_t>(loop[k + 1]);
                ++nt;
            }
        }
        t.ntri[cfg] = static_cast<uint8_t>(nt);
    }
    return t;
}

const McTable& mc_table() {
    static const McTable t = build_mc_table();
    return t;
}

// ---- kernels ----------------------------------------------------------------
struct MeshGeom {
    int r0, r1, r2;
    double lo0, lo1, lo2;
    double ext0, ext1, ext2;
    double sp0, sp1, sp2;
};

// binary64 points as load_frame makes them (:46-58): astype(float64), then
// (x, y, z) -> (x, z, y) when swap is set
__global__ __launch_bounds__(kMeshThreads) void k_mesh_points(const float* __restrict__ xyz, u64 n,
                                                              int swap, double* __restrict__ P) {
    const u64 i = static_cast<u64>(blockIdx.x) * kMeshThreads + threadIdx.x;
    if (i >= n) return;
    const double x = xyz[3 * i], y = xyz[3 * i + 1], z = xyz[3 * i + 2];
    P[3 * i] = x;
    P[3 * i + 1] = swap ? z : y;
    P[3 * i + 2] = swap ? y : z;
}

// Per-workgroup partials: min x, y, z, max x, y, z and the number of
// non-finite coordinates (fmin/fmax skip NaN, so the count is what lets the
// host refuse a point set holding one before any k-NN search runs).
constexpr int kBoundsPart = 7;
__global__ __launch_bounds__(kMeshThreads) void k_mesh_bounds(const double* __restrict__ P, u64 n,
                                                              double* __restrict__ part) {
    __shared__ double s[kBoundsPart][kMeshThreads / 64];
    double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    double bad = 0.0;
    const u64 stride = static_cast<u64>(gridDim.x) * kMeshThreads;
    for (u64 i = static_cast<u64>(blockIdx.x) * kMeshThreads + threadIdx.x; i < n; i += stride) {
        for (int a = 0; a < 3; ++a) {
            const double c = P[3 * i + a];
            mn[a] = fmin(mn[a], c);
            mx[a] = fmax(mx[a], c);
            bad += isfinite(c) ? 0.0 : 1.0;
        }
    }
    double v[kBoundsPart] = {mn[0], mn[1], mn[2], mx[0], mx[1], mx[2], bad};
#pragma unroll
    for (int k = 0; k < kBoundsPart; ++k)
        for (int o = 32; o > 0; o >>= 1) {
            const double u = __shfl_xor(v[k], o, 64);
            v[k] = k < 3 ? fmin(v[k], u) : k < 6 ? fmax(v[k], u) : v[k] + u;
        }
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < kBoundsPart; ++k) s[k][threadIdx.x >> 6] = v[k];
    __syncthreads();
    if (threadIdx.x < kBoundsPart) {
        double r = s[threadIdx.x][0];
        for (int k = 1; k < kMeshThreads / 64; ++k) {
            const double o = s[threadIdx.x][k];
            r = threadIdx.x < 3 ? fmin(r, o) : (threadIdx.x < 6 ? fmax(r, o) : r + o);
        }
        part[kBoundsPart * blockIdx.x + threadIdx.x] = r;
    }
}

// numpy's ((p - lo) / extent * res).astype(int), then clip to [0, res - 1]
__device__ __forceinline__ int voxel_of(double p, double lo, double ext, int res) {
    const double f = (p - lo) / ext * static_cast<double>(res);
    long long k = f == f ? static_cast<long long>(f) : 0;
    if (k < 0) k = 0;
    if (k > res - 1) k = res - 1;
    return static_cast<int>(k);
}

__global__ __launch_bounds__(kMeshThreads) void k_mesh_splat(const double* __restrict__ P, u64 n,
                                                             MeshGeom G, u32* __restrict__ count) {
    const u64 i = static_cast<u64>(blockIdx.x) * kMeshThreads + threadIdx.x;
    if (i >= n) return;
    const int a = voxel_of(P[3 * i], G.lo0, G.ext0, G.r0);
    const int b = voxel_of(P[3 * i + 1], G.lo1, G.ext1, G.r1);
    const int c = voxel_of(P[3 * i + 2], G.lo2, G.ext2, G.r2);
    atomicAdd(count + (static_cast<u64>(a) * G.r1 + b) * G.r2 + c, 1u);
}

// ---- k-nearest-neighbour position smoothing (smooth_positions_knn, :61-74)
// Each point becomes the mean of its k nearest points (itself included), in
// binary64, summed in ascending (distance^2, index) order and divided by k,
// as numpy's mean over cKDTree.query's rows.  Exact kNN on a uniform grid:
// rings of cells around the home cell are scanned until the k-th distance is
// below the ring's reach (points outside rings 0..R lie at least R cells away).

// A list that many waves append to, in kParts parts: one counter takes about
// 130 million atomics a second, 1 ms where 600,000 of a million points fall
// short of the guessed radius (k_knn_group on a splash: 1,314 -> 273 us with 64
// counters).  Workgroup t fills part t % kParts, and a consumer's workgroup reads one
// part and appends to the same part of its own lists, so a part holds no more
// than the items of its first producer's workgroups.
constexpr u32 kParts = 64;
constexpr u32 kPartLine = 16;  // counters apart by a cache line
constexpr u32 kPartCounts = kParts * kPartLine;
struct SplitList {
    u32* count;
    u32* items;
    u32 cap;  // of a part
    __device__ __forceinline__ u32 size(u32 part) const { return count[part * kPartLine]; }
    __device__ __forceinline__ u32 at(u32 part, u32 k) const {
        return items[static_cast<u64>(part) * cap + k];
    }
    // Appends q of every active lane, one atomic a wave.
    __device__ __forceinline__ void wave_append(u32 part, u32 q) const {
        const unsigned long long act = __ballot(1);
        const int first = __ffsll(act) - 1, lane = threadIdx.x & 63;
        u32 k = 0;
        if (lane == first)
            k = atomicAdd(count + part * kPartLine, static_cast<u32>(__popcll(act)));
        k = __shfl(k, first, 64) + static_cast<u32>(__popcll(act & ((1ull << lane) - 1ull)));
        items[static_cast<u64>(part) * cap + k] = q;
    }
};
// Capacity of a part when `blocks` workgroups append up to `per` items each.
inline u32 part_capacity(u64 blocks, u32 per) {
    return static_cast<u32>((blocks + kParts - 1) / kParts) * per;
}

struct KnnGrid {
    double lo0, lo1, lo2, cell;
    double guess;  // squared radius of about k + 4 points
    int d0, d1, d2;
};

__device__ __forceinline__ int knn_cell(double p, double lo, double cell, int d) {
    const double f = (p - lo) / cell;
    int k = f >= 0.0 ? static_cast<int>(f) : 0;
    return k > d - 1 ? d - 1 : k;
}

__global__ __launch_bounds__(kMeshThreads) void k_knn_keys(const double* __restrict__ P, u32 n,
                                                           KnnGrid g, u32* __restrict__ keys,
                                                           u32* __restrict__ vals) {
    const u32 i = blockIdx.x * kMeshThreads + threadIdx.x;
    if (i >= n) return;
    const int a = knn_cell(P[3ull * i], g.lo0, g.cell, g.d0);
    const int b = knn_cell(P[3ull * i + 1], g.lo1, g.cell, g.d1);
    const int c = knn_cell(P[3ull * i + 2], g.lo2, g.cell, g.d2);
    keys[i] = (static_cast<u32>(a) * g.d1 + b) * g.d2 + c;
    vals[i] = i;
}

// Points in cell order, so that a cell's candidates are read contiguously.
__global__ __launch_bounds__(kMeshThreads) void k_knn_gather(const double* __restrict__ P, u32 n,
                                                             const u32* __restrict__ sorted,
                                                             double* __restrict__ Ps) {
    const u32 s = blockIdx.x * kMeshThreads + threadIdx.x;
    if (s >= n) return;
    const u32 j = sorted[s];
    Ps[3ull * s] = P[3ull * j];
    Ps[3ull * s + 1] = P[3ull * j + 1];
    Ps[3ull * s + 2] = P[3ull * j + 2];
}

// Candidates s in [lo, hi) of the cell order into the ascending (d^2, id)
// list of the K nearest so far, the next candidate loaded while the current
// one is compared.
template <int K>
__device__ __forceinline__ void knn_scan(u32 lo, u32 hi, double px, double py, double pz,
                                         const double* __restrict__ Ps,
                                         const u32* __restrict__ sorted, double (&bd)[K],
                                         u32 (&bi)[K]) {
    if (lo >= hi) return;
    double nx = Ps[3ull * lo], ny = Ps[3ull * lo + 1], nz = Ps[3ull * lo + 2];
    u32 nj = sorted[lo];
    for (u32 s = lo; s < hi; ++s) {
        const double dx = nx - px, dy = ny - py, dz = nz - pz;
        u32 id = nj;
        if (s + 1 < hi) {
            nx = Ps[3ull * s + 3], ny = Ps[3ull * s + 4], nz = Ps[3ull * s + 5];
            nj = sorted[s + 1];
        }
        double d = (dx * dx + dy * dy) + dz * dz;
        // most candidates do not beat the current k-th: one test
        if (!(d < bd[K - 1] || (d == bd[K - 1] && id < bi[K - 1]))) continue;
        // insert (d, id) into the ascending list (compile-time indices)
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const bool less = d < bd[k] || (d == bd[k] && id < bi[k]);
            const double td = bd[k];
            const u32 ti = bi[k];
            bd[k] = less ? d : td;
            bi[k] = less ? id : ti;
            d = less ? td : d;
            id = less ? ti : id;
        }
    }
}

// Rings a lane walks on its own; points whose k-th neighbour lies further
// out go to a list that k_knn_far searches a wave per point.
constexpr int kKnnLaneRings = 3;

// Number of different keys among n sorted ones, added to *used.
__global__ __launch_bounds__(kMeshThreads) void k_knn_used(const u32* __restrict__ keys, u32 n,
                                                           u32* __restrict__ used) {
    u32 c = 0;
    for (u64 k = static_cast<u64>(blockIdx.x) * kMeshThreads + threadIdx.x; k < n;
         k += static_cast<u64>(gridDim.x) * kMeshThreads)
        c += k == 0 || keys[k] != keys[k - 1] ? 1u : 0u;
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(used, c);
}

template <int K>
__device__ __forceinline__ void knn_lane(const double* __restrict__ P, KnnGrid g,
                                         const u32* __restrict__ sorted,
                                         const double* __restrict__ Ps,
                                         const u32* __restrict__ cs, double* __restrict__ out,
                                         const SplitList& far, u32 part, u32 q) {
    const u32 i = sorted[q];
    const double px = Ps[3ull * q], py = Ps[3ull * q + 1], pz = Ps[3ull * q + 2];
    const int h0 = knn_cell(px, g.lo0, g.cell, g.d0);
    const int h1 = knn_cell(py, g.lo1, g.cell, g.d1);
    const int h2 = knn_cell(pz, g.lo2, g.cell, g.d2);
    double bd[K];
    u32 bi[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        bd[k] = INFINITY;
        bi[k] = 0xFFFFFFFFu;
    }
    auto scan = [&](u32 lo, u32 hi) { knn_scan<K>(lo, hi, px, py, pz, Ps, sorted, bd, bi); };
    const int rmax = max(g.d0, max(g.d1, g.d2));
    const int rlim = min(rmax, kKnnLaneRings);
    bool done = false;
    for (int R = 0; R <= rlim; ++R) {
        const int c0 = max(h2 - R, 0), c1 = min(h2 + R, g.d2 - 1);
        for (int a = max(h0 - R, 0); a <= min(h0 + R, g.d0 - 1); ++a) {
            for (int b = max(h1 - R, 0); b <= min(h1 + R, g.d1 - 1); ++b) {
                const u32 row = (static_cast<u32>(a) * g.d1 + b) * g.d2;
                if (R == 0 || a == h0 - R || a == h0 + R || b == h1 - R || b == h1 + R) {
                    // a face of the shell: the whole row, one contiguous range
                    scan(cs[row + c0], cs[row + c1 + 1]);
                } else {  // inside the shell's faces: its two ends in c
                    if (h2 - R >= 0) scan(cs[row + h2 - R], cs[row + h2 - R + 1]);
                    if (h2 + R < g.d2) scan(cs[row + h2 + R], cs[row + h2 + R + 1]);
                }
            }
        }
        const double reach = static_cast<double>(R) * g.cell * (1.0 - 1e-9);
        if (bi[K - 1] != 0xFFFFFFFFu && bd[K - 1] < reach * reach) {
            done = true;
            break;
        }
    }
    if (!done && rlim < rmax) {  // rings beyond rlim hold cells: leave it to k_knn_far
        far.wave_append(part, q);
        return;
    }
    double sx = 0.0, sy = 0.0, sz = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const u32 j = bi[k];
        if (j == 0xFFFFFFFFu) continue;  // never with finite input (the host refuses others)
        sx = sx + P[3ull * j];
        sy = sy + P[3ull * j + 1];
        sz = sz + P[3ull * j + 2];
    }
    out[3ull * i] = sx / static_cast<double>(K);
    out[3ull * i + 1] = sy / static_cast<double>(K);
    out[3ull * i + 2] = sz / static_cast<double>(K);
}

// One thread per listed point (dense or far neighbourhoods that
// k_knn_group leaves).
template <int K>
__global__ __launch_bounds__(kMeshThreads) void k_knn_smooth(
    const double* __restrict__ P, KnnGrid g, const u32* __restrict__ sorted,
    const double* __restrict__ Ps, const u32* __restrict__ cs, SplitList list,
    double* __restrict__ out, SplitList far) {
    const u32 part = blockIdx.x % kParts, n = list.size(part);
    const u32 stride = gridDim.x / kParts * kMeshThreads;
    for (u32 k = blockIdx.x / kParts * kMeshThreads + threadIdx.x; k < n; k += stride)
        knn_lane<K>(P, g, sorted, Ps, cs, out, far, part, list.at(part, k));
}

// G lanes per point over the rings 0..R at once.  A lane that keeps the K
// nearest of all candidates in registers spends its time on the insertion (15
// steps of binary64 compares whenever any lane of the wave accepts) and
// leaves small clouds to one wave per CU.  Here the group splits the
// candidates, lists those within a limit in LDS (a few more than K), each
// listed point finds its rank among them, and the K first are summed in
// ascending (d^2, id) order, one lane per coordinate.  The limit is
//   GUESS: g.guess, the squared radius that holds about K + 4 points at the
//     expected spacing, in one visit of the candidates;
//   else: the first of kKnnBins bins of [0, reach^2) at which K points are
//     counted, in two visits; where that bin brings more than the list holds
//     (dense spots), the bins of the range up to it, and so on.
// Either way it lies below the reach, the point's own distance to the faces
// of the scanned block (none where the block ends the grid).  Points with
// fewer than K neighbours in the limit go to `few`, with more than the list
// holds to `many`.  A pass over 1,001,385 points, 15 neighbours, with the
// guess: 312 us with 8 lanes, 412 with 4, 403 with 16 (one lane a point:
// 1,267); 17,056 points: 18 us with 8 lanes (256).  Bins in both visits for
// every point: 799 us.  Two passes over 30,000 points at a sixth of the expected
// spacing among 10,648 others, ms: narrowing 10.7, without (one lane a point
// for those) 29, one lane for every point 13.3.
constexpr int kKnnBins = 32;
constexpr u32 kKnnLong = 512;  // candidates of a row (three cells of about k / 3 points)
constexpr int kKnnRounds = 6;  // a round narrows the range to an eighth or less where it helps
constexpr int kKnnLists = 5;  // of points, between the passes of knn_pass
constexpr int knn_cap(int k) { return k <= 16 ? 32 : 64; }  // listed points
template <int K, int R, int G, bool GUESS>
__global__ __launch_bounds__(kMeshThreads) void k_knn_group(
    u32 n, SplitList list, KnnGrid g, const u32* __restrict__ sorted,
    const double* __restrict__ Ps, const u32* __restrict__ cs, double* __restrict__ out,
    SplitList few, SplitList many) {
    constexpr u32 kCap = knn_cap(K);
    static_assert(K <= kCap && kCap <= 256, "list holds the K nearest, places in 8 bits");
    constexpr int W = 2 * R + 1, kRows = W * W;
    constexpr int kPts = kMeshThreads / G;
    __shared__ u32 s_lo[kPts][kRows], s_hi[kPts][kRows];
    __shared__ u32 s_bin[GUESS ? 1 : kPts][kKnnBins / 2];  // two 16-bit counts a word
    __shared__ u32 s_cnt[kPts];
    __shared__ double s_d[kPts][kCap];
    __shared__ u32 s_slot[kPts][kCap];
    __shared__ uint8_t s_ord[kPts][K];
    const int pt = threadIdx.x / G, lane = threadIdx.x % G;
    // GUESS takes all points, a tile of kPts after the other, the others a part
    // of their list
    const u32 own = blockIdx.x % kParts;
    const u32 total = GUESS ? n : list.size(own);
    const u32 stride = (GUESS ? gridDim.x : gridDim.x / kParts) * kPts;
    // LDS below is private to the group, whose lanes share a wave
    auto sync = [] { wave_lds_sync(); };
    for (u32 f = (GUESS ? blockIdx.x : blockIdx.x / kParts) * kPts + pt; f < total; f += stride) {
        const u32 q = GUESS ? f : list.at(own, f);
        const double px = Ps[3ull * q], py = Ps[3ull * q + 1], pz = Ps[3ull * q + 2];
        const int h0 = knn_cell(px, g.lo0, g.cell, g.d0);
        const int h1 = knn_cell(py, g.lo1, g.cell, g.d1);
        const int h2 = knn_cell(pz, g.lo2, g.cell, g.d2);
        const int c0 = max(h2 - R, 0), c1 = min(h2 + R, g.d2 - 1);
        sync();  // (the point before may have ended at a continue)
        if (lane == 0) s_cnt[pt] = 0;
        sync();
        for (int r = lane; r < kRows; r += G) {
            const int a = h0 - R + r / W, b = h1 - R + r % W;
            const bool in = a >= 0 && a < g.d0 && b >= 0 && b < g.d1;
            const u32 row = in ? (static_cast<u32>(a) * g.d1 + b) * g.d2 : 0u;
            const u32 first = in ? cs[row + c0] : 0u, end = in ? cs[row + c1 + 1] : 0u;
            s_lo[pt][r] = first;
            s_hi[pt][r] = end;
            // forty times the expected points: not a place for the guess
            if (GUESS && end - first > kKnnLong) s_cnt[pt] = kCap + 1;
        }
        // distance to the faces of the scanned block that other cells touch
        double reach = INFINITY;
        auto face = [&](double p, double lo, int h, int d) {
            if (h - R > 0) reach = fmin(reach, p - (lo + (h - R) * g.cell));
            if (h + R < d - 1) reach = fmin(reach, (lo + (h + R + 1) * g.cell) - p);
        };
        face(px, g.lo0, h0, g.d0);
        face(py, g.lo1, h1, g.d1);
        face(pz, g.lo2, h2, g.d2);
        const bool all = reach == INFINITY;  // the block is the whole grid
        if (all) {  // every candidate lies within the grid's diagonal
            const double a = g.d0 * g.cell, b = g.d1 * g.cell, c = g.d2 * g.cell;
            reach = 1.1 * sqrt(a * a + b * b + c * c);
        }
        reach = fmax(reach * (1.0 - 1e-9), 0.0);
        // the group shares every row, or with many rows each lane takes its own
        constexpr bool kOwnRows = R > 2;
        auto visit = [&](auto&& use) {
            for (int r = kOwnRows ? lane : 0; r < kRows; r += kOwnRows ? G : 1) {
                const u32 hi = s_hi[pt][r];
                for (u32 s = s_lo[pt][r] + (kOwnRows ? 0 : lane); s < hi; s += kOwnRows ? 1 : G) {
                    const double dx = Ps[3ull * s] - px, dy = Ps[3ull * s + 1] - py,
                                 dz = Ps[3ull * s + 2] - pz;
                    use(s, (dx * dx + dy * dy) + dz * dz);
                }
            }
        };
        auto append = [&](u32 s, double d) {
            const u32 k = atomicAdd(&s_cnt[pt], 1u);
            if (k < kCap) {
                s_d[pt][k] = d;
                s_slot[pt][k] = s;
            }
        };
        u32 m = 0;  // listed points
        bool overfull = false;
        if constexpr (GUESS) {
            const double lim = fmin(g.guess, reach * reach);
            sync();
            const bool crowded = s_cnt[pt] != 0;
            sync();
            if (!crowded)
                visit([&](u32 s, double d) {
                    if (d < lim) append(s, d);
                });
            sync();
            m = s_cnt[pt];
        } else {
            sync();
            u32 have = 0;
            for (int r = 0; r < kRows; ++r) have += s_hi[pt][r] - s_lo[pt][r];
            overfull = have > 0xFFFFu;
            double span = reach * reach;  // the bins' range
            float scale = 0.0f;
            int top = -1;  // last bin of the list
            u32 last = 0;
            for (int round = 0; !overfull && round < kKnnRounds; ++round) {
                for (int k = lane; k < kKnnBins / 2; k += G) s_bin[pt][k] = 0;
                sync();
                scale = span > 0.0 ? static_cast<float>(static_cast<double>(kKnnBins) / span)
                                   : INFINITY;
                // the bin is monotone in d; the last one of the whole range
                // may miss points beyond the block and never counts
                const int bins = round == 0 ? kKnnBins - 1 : kKnnBins;
                u32 same = 0;
                visit([&](u32, double d) {
                    same += d == 0.0 ? 1u : 0u;
                    const float bin = static_cast<float>(d) * scale;
                    if (bin < static_cast<float>(bins)) {
                        const u32 b = static_cast<u32>(bin);
                        atomicAdd(&s_bin[pt][b >> 1], b & 1u ? 0x10000u : 1u);
                    }
                });
                if (same) atomicAdd(&s_cnt[pt], same);
                sync();
                // more points at one place than the list holds: no bins part them
                overfull = s_cnt[pt] > kCap;
                sync();
                if (lane == 0) s_cnt[pt] = 0;
                m = 0;
#pragma unroll
                for (int b = 0; b < kKnnBins; ++b) {
                    const u32 c = (s_bin[pt][b >> 1] >> (16 * (b & 1))) & 0xFFFFu;
                    if (m < static_cast<u32>(K)) {
                        m += c;
                        top = b;
                    }
                }
                sync();
                // a dense spot: the same again over the bins up to there, while
                // that tells the points apart
                if (m <= kCap || m == last) break;
                last = m;
                span *= static_cast<double>(top + 1) / static_cast<double>(kKnnBins);
            }
            if (m >= static_cast<u32>(K) && m <= kCap) {
                const float lim = static_cast<float>(top + 1);
                visit([&](u32 s, double d) {
                    if (static_cast<float>(d) * scale < lim) append(s, d);
                });
                sync();
            }
        }
        if (overfull || m < static_cast<u32>(K) || m > kCap) {
            if (lane == 0) {
                const u32 part = GUESS ? f / kPts % kParts : own;
                if (!overfull && m < static_cast<u32>(K)) few.wave_append(part, q);
                else many.wave_append(part, q);
            }
            continue;
        }
        for (u32 e = lane; e < m; e += G) {
            const double d = s_d[pt][e];
            u32 rank = 0, tied = 0;
            for (u32 k = 0; k < m; ++k) {
                const double o = s_d[pt][k];
                rank += o < d ? 1u : 0u;
                tied += o == d ? 1u : 0u;  // itself included
            }
            if (tied > 1u && rank < static_cast<u32>(K)) {  // lower ids first
                const u32 id = sorted[s_slot[pt][e]];
                for (u32 k = 0; k < m; ++k)
                    if (s_d[pt][k] == d && sorted[s_slot[pt][k]] < id) ++rank;
            }
            if (rank < static_cast<u32>(K)) s_ord[pt][rank] = static_cast<uint8_t>(e);
        }
        sync();
        if (lane < 3) {
            double v[K];
#pragma unroll
            for (int k = 0; k < K; ++k) v[k] = Ps[3ull * s_slot[pt][s_ord[pt][k]] + lane];
            double sum = 0.0;
#pragma unroll
            for (int k = 0; k < K; ++k) sum = sum + v[k];
            out[3ull * sorted[q] + lane] = sum / static_cast<double>(K);
        }
        sync();
    }
}

// The listed points, one wave each: the lanes take the (a, b) rows of every
// shell in turn, each keeping the K nearest of its own rows; the shells stop
// once K candidates of the union lie inside the reach (then the union's K-th
// does), and K rounds of the wave minimum by (d^2, id) give the K nearest in
// ascending order for the sum.
template <int K>
__global__ __launch_bounds__(kMeshThreads) void k_knn_far(const double* __restrict__ P,
                                                          KnnGrid g,
                                                          const u32* __restrict__ sorted,
                                                          const double* __restrict__ Ps,
                                                          const u32* __restrict__ cs,
                                                          SplitList far,
                                                          double* __restrict__ out) {
    const int lane = threadIdx.x & 63;
    const u32 part = blockIdx.x % kParts, nfar = far.size(part);
    const u32 wave = (blockIdx.x / kParts * kMeshThreads + threadIdx.x) >> 6;
    const u32 nwaves = (gridDim.x / kParts * kMeshThreads) >> 6;
    const int rmax = max(g.d0, max(g.d1, g.d2));
    for (u32 f = wave; f < nfar; f += nwaves) {
        const u32 q = far.at(part, f);
        const double px = Ps[3ull * q], py = Ps[3ull * q + 1], pz = Ps[3ull * q + 2];
        const int h0 = knn_cell(px, g.lo0, g.cell, g.d0);
        const int h1 = knn_cell(py, g.lo1, g.cell, g.d1);
        const int h2 = knn_cell(pz, g.lo2, g.cell, g.d2);
        double bd[K];
        u32 bi[K];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            bd[k] = INFINITY;
            bi[k] = 0xFFFFFFFFu;
        }
        for (int R = 0; R <= rmax; ++R) {
            // the shell's (a, b) rows inside the grid: na * nb <= d0 * d1 <= 2^26
            const int a0 = max(h0 - R, 0), na = min(h0 + R, g.d0 - 1) - a0 + 1;
            const int b0 = max(h1 - R, 0), nb = min(h1 + R, g.d1 - 1) - b0 + 1;
            const int c0 = max(h2 - R, 0), c1 = min(h2 + R, g.d2 - 1);
            for (int t = lane; t < na * nb; t += 64) {
                const int a = a0 + t / nb, b = b0 + t % nb;
                const u32 row = (static_cast<u32>(a) * g.d1 + b) * g.d2;
                if (R == 0 || a == h0 - R || a == h0 + R || b == h1 - R || b == h1 + R) {
                    knn_scan<K>(cs[row + c0], cs[row + c1 + 1], px, py, pz, Ps, sorted, bd, bi);
                } else {
                    if (h2 - R >= 0)
                        knn_scan<K>(cs[row + h2 - R], cs[row + h2 - R + 1], px, py, pz, Ps,
                                    sorted, bd, bi);
                    if (h2 + R < g.d2)
                        knn_scan<K>(cs[row + h2 + R], cs[row + h2 + R + 1], px, py, pz, Ps,
                                    sorted, bd, bi);
                }
            }
            const double reach = static_cast<double>(R) * g.cell * (1.0 - 1e-9);
            u32 inside = 0;
#pragma unroll
            for (int k = 0; k < K; ++k) inside += bd[k] < reach * reach ? 1u : 0u;
            for (int o = 32; o > 0; o >>= 1) inside += __shfl_xor(inside, o, 64);
            if (inside >= static_cast<u32>(K)) break;  // the same on every lane
        }
        double sx = 0.0, sy = 0.0, sz = 0.0;
        for (int r = 0; r < K; ++r) {
            double d = bd[0];
            u32 id = bi[0];
            for (int o = 32; o > 0; o >>= 1) {
                const double od = __shfl_xor(d, o, 64);
                const u32 oi = __shfl_xor(id, o, 64);
                if (od < d || (od == d && oi < id)) {
                    d = od;
                    id = oi;
                }
            }
            // every candidate sits in one lane's list: its owner pops it
            const bool mine = bi[0] == id;
#pragma unroll
            for (int k = 0; k + 1 < K; ++k) {
                bd[k] = mine ? bd[k + 1] : bd[k];
                bi[k] = mine ? bi[k + 1] : bi[k];
            }
            bd[K - 1] = mine ? INFINITY : bd[K - 1];
            bi[K - 1] = mine ? 0xFFFFFFFFu : bi[K - 1];
            if (id != 0xFFFFFFFFu) {  // always, with finite input
                sx = sx + P[3ull * id];
                sy = sy + P[3ull * id + 1];
                sz = sz + P[3ull * id + 2];
            }
        }
        if (lane == 0) {
            const u32 i = sorted[q];
            out[3ull * i] = sx / static_cast<double>(K);
            out[3ull * i + 1] = sy / static_cast<double>(K);
            out[3ull * i + 2] = sz / static_cast<double>(K);
        }
    }
}

__global__ __launch_bounds__(kMeshThreads) void k_mesh_to_float(const u32* __restrict__ count,
                                                                float* __restrict__ grid, u64 nv) {
    const u64 i = static_cast<u64>(blockIdx.x) * kMeshThreads + threadIdx.x;
    if (i < nv) grid[i] = static_cast<float>(count[i]);
}

// scipy.ndimage 'reflect' extension: (d c b a | a b c d | d c b a), repeated
__device__ __forceinline__ int reflect_index(int k, int n) {
    const int p = 2 * n;
    k %= p;
    if (k < 0) k += p;
    return k >= n ? p - 1 - k : k;
}

// One 1-D pass along `axis` with 2R+1 symmetric weights w (w[R] the centre):
// acc = x[i] w[R] + sum_{j=1..R} (x[i-j] + x[i+j]) w[R+j] in binary64.
__global__ __launch_bounds__(kMeshThreads) void k_mesh_blur(const float* __restrict__ in,
                                                            float* __restrict__ out, int r0, int r1,
                                                            int r2, int axis,
                                                            const double* __restrict__ w, int R) {
    const u64 nv = static_cast<u64>(r0) * r1 * r2;
    const u64 i = static_cast<u64>(blockIdx.x) * kMeshThreads + threadIdx.x;
    if (i >= nv) return;
    const int c = static_cast<int>(i % r2);
    const int b = static_cast<int>((i / r2) % r1);
    const int a = static_cast<int>(i / (static_cast<u64>(r2) * r1));
    int pos, len;
    u64 step;
    if (axis == 0) {
        pos = a, len = r0, step = static_cast<u64>(r1) * r2;
    } else if (axis == 1) {
        pos = b, len = r1, step = static_cast<u64>(r2);
    } else {
        pos = c, len = r2, step = 1;
    }
    const u64 base = i - static_cast<u64>(pos) * step;
    double acc = static_cast<double>(in[i]) * w[R];
    if (pos >= R && pos + R < len) {  // no reflection: consecutive taps
        for (int j = 1; j <= R; ++j) {
            const double lo = in[i - static_cast<u64>(j) * step];
            const double hi = in[i + static_cast<u64>(j) * step];
            acc += (lo + hi) * w[R + j];
        }
    } else {
        for (int j = 1; j <= R; ++j) {
            const double lo = in[base + static_cast<u64>(reflect_index(pos - j, len)) * step];
            const double hi = in[base + static_cast<u64>(reflect_index(pos + j, len)) * step];
            acc += (lo + hi) * w[R + j];
        }
    }
    out[i] = static_cast<float>(acc);
}

// Tiled blur passes.  A strided pass (axis 1 over each (b, c) plane, rows of
// r2 values; axis 0 over the whole grid, rows of r1 r2 values, so its tiles
// need not end with a row of c) stages, per workgroup, 64 consecutive
// columns x (kBlurTile + 2R) positions along the axis in LDS,
// with the 'reflect' ends resolved while loading, so every input is read from
// HBM about (kBlurTile + 2R) / kBlurTile times instead of 2R + 1 times; each
// of the 4 wave rows then forms kBlurTile / 4 outputs, taps outermost so each
// weight is loaded once.  Sums and their order are k_mesh_blur's.
constexpr int kBlurTile = 64;
constexpr int kBlurMaxR = 64;  // LDS (kBlurTile + 2R) x 64 floats, 48 KiB at most

__device__ __forceinline__ float blur_in(const float* p, u64 i) { return p[i]; }
__device__ __forceinline__ float blur_in(const u32* p, u64 i) { return static_cast<float>(p[i]); }

// position k of an axis of length n, 'reflect' beyond the ends
__device__ __forceinline__ int reflect_fast(int k, int n) {
    return k >= 0 && k < n ? k : reflect_index(k, n);
}

// RT > 0: a tap radius R <= RT at compile time.  Each thread then widens its
// kBlurTile / 4 + 2 RT inputs once and keeps them in registers for all taps,
// instead of two LDS reads and two conversions per tap and output; the taps
// between R and RT have weight 0 and add +0 (80.5 million voxels, R = 10:
// axis 0 385 -> 273 us, axis 1 343 -> 207 us).
template <typename In, int RT>
__global__ __launch_bounds__(256) void k_blur_strided(const In* __restrict__ in,
                                                      float* __restrict__ out, u32 width, int len,
                                                      u64 plane, const double* __restrict__ w,
                                                      int Rrt) {
    const int R = RT > 0 ? RT : Rrt;
    extern __shared__ float sb[];  // [(kBlurTile + 2R) * 64]
    const int lx = threadIdx.x & 63, ly = threadIdx.x >> 6;
    const u32 c = blockIdx.x * 64 + lx;  // column of the plane: < width
    const int p0 = blockIdx.y * kBlurTile;
    const u64 step = width;
    const u64 base = blockIdx.z * plane + c;  // position 0 of this column
    const bool cin = c < width;
    const int rows = kBlurTile + 2 * R;
    if constexpr (RT > 0) {
        // every load of a thread in flight before its first LDS store
        constexpr int N = (kBlurTile + 2 * RT) / 4;
        static_assert((kBlurTile + 2 * RT) % 4 == 0, "whole rounds of rows");
        float v[N];
#pragma unroll
        for (int k = 0; k < N; ++k)
            v[k] = cin ? blur_in(in, base + static_cast<u64>(reflect_fast(p0 - R + ly + 4 * k, len)) *
                                                step)
                       : 0.0f;
#pragma unroll
        for (int k = 0; k < N; ++k) sb[(ly + 4 * k) * 64 + lx] = v[k];
    } else {
        for (int k = ly; k < rows; k += 4)
            sb[k * 64 + lx] =
                cin ? blur_in(in, base + static_cast<u64>(reflect_fast(p0 - R + k, len)) * step)
                    : 0.0f;
    }
    __syncthreads();
    constexpr int M = kBlurTile / 4;
    double acc[M];
    if constexpr (RT > 0) {
        double x[M + 2 * RT];
        const float* col = sb + ly * M * 64 + lx;
#pragma unroll
        for (int k = 0; k < M + 2 * RT; ++k) x[k] = static_cast<double>(col[k * 64]);
        const double w0 = w[RT];
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] = x[m + RT] * w0;
#pragma unroll
        for (int j = 1; j <= RT; ++j) {
            const double wj = w[RT + j];
#pragma unroll
            for (int m = 0; m < M; ++m) acc[m] += (x[m + RT - j] + x[m + RT + j]) * wj;
        }
    } else {
        const double w0 = w[R];
#pragma unroll
        for (int m = 0; m < M; ++m)
            acc[m] = static_cast<double>(sb[(ly * M + m + R) * 64 + lx]) * w0;
        for (int j = 1; j <= R; ++j) {
            const double wj = w[R + j];
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int k = ly * M + m + R;
                acc[m] += (static_cast<double>(sb[(k - j) * 64 + lx]) +
                           static_cast<double>(sb[(k + j) * 64 + lx])) * wj;
            }
        }
    }
    if (!cin) return;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int p = p0 + ly * M + m;
        if (p < len) out[base + static_cast<u64>(p) * step] = static_cast<float>(acc[m]);
    }
}

// The contiguous pass (axis 2): each wave takes kBlurRows (a, b) rows in turn,
// 256 consecutive c plus 2R halo in LDS at a time, four consecutive outputs
// per lane (the inputs read as 16-byte words and widened once: 80.5 million
// voxels, R = 10, 375 -> 215 us), and the workgroup writes the maximum of
// its outputs to part[] (blurred densities are >= 0, so 0 is neutral).
// RT > 0: a tap radius R <= RT at compile time (weight 0 beyond R); RT == 0
// takes R, one tap after the other from LDS, a lane's outputs 64 apart so that
// the reads of a tap hit different banks (17.6 million voxels, R = 40: a
// workgroup per row 367 us, outputs side by side 650, 64 apart 212).
constexpr int kBlurRows = 4;  // (a, b) rows per wave of the contiguous pass
constexpr int kBlurSeg = 256;
__host__ __device__ constexpr int blur_row_floats(int R) { return (kBlurSeg + 2 * R + 3) / 4 * 4; }

template <int RT>
__global__ __launch_bounds__(256) void k_blur_rows(const float* __restrict__ in,
                                                   float* __restrict__ out, u64 rows, int r2,
                                                   const double* __restrict__ w, int Rrt,
                                                   float* __restrict__ part) {
    const int R = RT > 0 ? RT : Rrt;
    extern __shared__ __align__(16) float sb[];  // one row segment per wave
    __shared__ float wmax[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float* const seg = sb + wave * blur_row_floats(R);
    float vmax = 0.0f;
    const u64 first = (static_cast<u64>(blockIdx.x) * 4 + wave) * kBlurRows;
    const u64 last = min(first + kBlurRows, rows);
    // the wave's own LDS: its instructions stay in order
    auto sync = [] { wave_lds_sync(); };
    // RT > 0: the next segment's loads are in flight while this one is summed
    constexpr int kLoads = RT > 0 ? (kBlurSeg + 2 * RT + 63) / 64 : 1;
    float ahead[kLoads];
    auto request = [&](u64 r, int c0) {
        const u64 row = r * r2;
#pragma unroll
        for (int u = 0; u < kLoads; ++u)
            ahead[u] = in[row + reflect_fast(min(c0 - R + lane + 64 * u, c0 + kBlurSeg + R - 1), r2)];
    };
    if constexpr (RT > 0)
        if (first < last) request(first, 0);
    for (u64 r = first; r < last; ++r) {
        const u64 row = r * r2;
        for (int c0 = 0; c0 < r2; c0 += kBlurSeg) {
            sync();
            if constexpr (RT > 0) {
#pragma unroll
                for (int u = 0; u < kLoads; ++u)
                    if (lane + 64 * u < blur_row_floats(RT)) seg[lane + 64 * u] = ahead[u];
                const bool more = c0 + kBlurSeg < r2;
                if (more || r + 1 < last) request(more ? r : r + 1, more ? c0 + kBlurSeg : 0);
            } else {
                for (int k = lane; k < kBlurSeg + 2 * R; k += 64)
                    seg[k] = in[row + reflect_fast(c0 - R + k, r2)];
            }
            sync();
            double acc[4];
            if constexpr (RT > 0) {
                constexpr int N = (4 + 2 * RT + 3) / 4 * 4;
                double x[N];
#pragma unroll
                for (int k = 0; k < N; k += 4) {
                    // the last lane's padding lies inside the segment's
                    const float4 f = *reinterpret_cast<const float4*>(seg + 4 * lane + k);
                    x[k] = f.x, x[k + 1] = f.y, x[k + 2] = f.z, x[k + 3] = f.w;
                }
#pragma unroll
                for (int m = 0; m < 4; ++m) acc[m] = x[m + RT] * w[RT];
#pragma unroll
                for (int j = 1; j <= RT; ++j) {
                    const double wj = w[RT + j];
#pragma unroll
                    for (int m = 0; m < 4; ++m) acc[m] += (x[m + RT - j] + x[m + RT + j]) * wj;
                }
            } else if (r2 - c0 > 64) {
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    acc[m] = static_cast<double>(seg[lane + 64 * m + R]) * w[R];
                for (int j = 1; j <= R; ++j) {
                    const double wj = w[R + j];
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const int k = lane + 64 * m + R;
                        acc[m] += (static_cast<double>(seg[k - j]) + static_cast<double>(seg[k + j])) * wj;
                    }
                }
            } else {  // one output per lane: narrow rows, ends of rows
                const int k = lane + R;
                acc[0] = static_cast<double>(seg[k]) * w[R];
                for (int j = 1; j <= R; ++j)
                    acc[0] += (static_cast<double>(seg[k - j]) + static_cast<double>(seg[k + j])) *
                              w[R + j];
                acc[1] = acc[2] = acc[3] = 0.0;  // past the row
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                const int c = c0 + (RT > 0 ? 4 * lane + m : lane + 64 * m);
                const float v = static_cast<float>(acc[m]);
                if (c < r2) {
                    out[row + c] = v;
                    vmax = fmaxf(vmax, v);
                }
            }
        }
    }
    for (int o = 32; o > 0; o >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, o, 64));
    if (lane == 0) wmax[wave] = vmax;
    __syncthreads();
    if (threadIdx.x == 0)
        part[blockIdx.x] = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
}

__global__ __launch_bounds__(kMeshThreads) void k_mesh_max(const float* __restrict__ g, u64 nv,
                                                           float* __restrict__ part) {
    __shared__ float s[kMeshThreads / 64];
    float m = -INFINITY;
    const u64 stride = static_cast<u64>(gridDim.x) * kMeshThreads;
    for (u64 i = static_cast<u64>(blockIdx.x) * kMeshThreads + threadIdx.x; i < nv; i += stride)
        m = fmaxf(m, g[i]);
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int k = 1; k < kMeshThreads / 64; ++k) m = fmaxf(m, s[k]);
        part[blockIdx.x] = m;
    }
}

struct McDev {
    uint8_t ntri[256];
    uint8_t tri[256][kMaxTri * 3];
};

// Marching cubes over segments: 64 consecutive c of one (a, b) row.  Segments
// in linear order cover the grid in grid-point order, so an exclusive scan of
// per-segment counts plus a prefix across the segment numbers every vertex by
// (grid point, axis) and every triangle by (cube, table order).  A grid point
// owns the crossing edges from it along +a, +b, +c (edge mask bits 0, 1, 2); a
// cube starts at its lowest corner.
//
// The grid is read once, into one inside bit per point (k_mc_bits).  Crossing
// edges and cube configurations then come from the 64-bit words of a segment
// and its neighbours: a thread per segment counts (k_mc_count), a thread per
// vertex and per cube with triangles emits (k_mc_vertices, k_mc_triangles).
struct McGrid {
    int r0, r1, r2;
    u32 ntx;    // segments per row
    u32 nseg;
    const u64* bits;
};

// Inside bits, eight segments per wave with their loads in flight together.
__global__ __launch_bounds__(256) void k_mc_bits(const float* __restrict__ g, u32 nseg, int r2,
                                                 u32 ntx, float iso, u64* __restrict__ bits) {
    constexpr u32 U = 8;
    const u32 lane = threadIdx.x & 63;
    const u32 wave = static_cast<u32>(
        __builtin_amdgcn_readfirstlane(static_cast<int>(blockIdx.x * 4 + (threadIdx.x >> 6))));
    for (u32 s0 = wave * U; s0 < nseg; s0 += gridDim.x * 4 * U) {
        float v[U];
#pragma unroll
        for (u32 u = 0; u < U; ++u) {
            const u32 row = (s0 + u) / ntx;
            const u32 c = (s0 + u - row * ntx) * 64u + lane;
            v[u] = s0 + u < nseg && c < static_cast<u32>(r2)
                       ? g[static_cast<u64>(row) * static_cast<u32>(r2) + c]
                       : -INFINITY;
        }
#pragma unroll
        for (u32 u = 0; u < U; ++u) {
            const u64 m = __ballot(v[u] > iso);
            if (lane == u && s0 + u < nseg) bits[s0 + u] = m;
        }
    }
}

// The words of segment s and of its neighbours that its edges and cubes read:
// row[k] and the same points one further along c (cnext[k]), k = da + 2 db;
// rows beyond the grid read 0.
struct McWords {
    u64 row[4], cnext[4];
    u64 valid, cvalid;  // points of the segment; those with a point at c + 1
    bool an, bn;        // a + 1, b + 1 inside the grid
    u32 a, b, tx;
    __device__ __forceinline__ McWords(const McGrid& M, u32 s) {
        const u32 r = s / M.ntx;
        tx = s - r * M.ntx;
        a = r / static_cast<u32>(M.r1);
        b = r - a * static_cast<u32>(M.r1);
        an = a + 1 < static_cast<u32>(M.r0);
        bn = b + 1 < static_cast<u32>(M.r1);
        const u32 left = static_cast<u32>(M.r2) - tx * 64u;  // points from here to the row's end
        valid = left >= 64u ? ~0ull : (1ull << left) - 1ull;
        cvalid = left > 64u ? ~0ull : (1ull << (left - 1u)) - 1ull;
        const bool tn = tx + 1 < M.ntx;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const bool in = (!(k & 1) || an) && (!(k & 2) || bn);
            const u32 t = s + ((k & 1) ? static_cast<u32>(M.r1) * M.ntx : 0u) + ((k & 2) ? M.ntx : 0u);
            row[k] = in ? M.bits[t] : 0ull;
            const u64 nx = in && tn ? M.bits[t + 1] : 0ull;
            cnext[k] = (row[k] >> 1) | (nx << 63);
        }
    }
    // crossing edges along axis 0, 1, 2
    __device__ __forceinline__ u64 edges(int axis) const {
        if (axis == 0) return an ? (row[0] ^ row[1]) & valid : 0ull;
        if (axis == 1) return bn ? (row[0] ^ row[2]) & valid : 0ull;
        return (row[0] ^ cnext[0]) & cvalid;
    }
    // cubes with corners on both sides
    __device__ __forceinline__ u64 cubes() const {
        if (!an || !bn) return 0ull;
        u64 any = 0ull, all = ~0ull;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            any |= row[k] | cnext[k];
            all &= row[k] & cnext[k];
        }
        return any & ~all & cvalid;
    }
    // configuration of the cube at bit c: corner k at (k & 1, k >> 1 & 1, k >> 2)
    __device__ __forceinline__ u32 config(u32 c) const {
        u32 cfg = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            cfg |= static_cast<u32>((row[k] >> c) & 1ull) << k;
            cfg |= static_cast<u32>((cnext[k] >> c) & 1ull) << (k + 4);
        }
        return cfg;
    }
};

// Counts of kScanBlock segments and their exclusive scan within the block:
// vertices, triangles and cubes with triangles, packed in one word.
constexpr int kScanBlock = kMeshThreads;
constexpr int kTriShift = 24, kCubeShift = 48;  // 192, 320 and 64 per segment at most
__device__ __forceinline__ u32 scan_verts(u64 v) { return static_cast<u32>(v) & 0xFFFFFFu; }
__device__ __forceinline__ u32 scan_tris(u64 v) { return static_cast<u32>(v >> kTriShift) & 0xFFFFFFu; }
__device__ __forceinline__ u32 scan_cubes(u64 v) { return static_cast<u32>(v >> kCubeShift); }

__global__ __launch_bounds__(kMeshThreads) void k_mc_count(McGrid M, const McDev* __restrict__ T,
                                                           u64* __restrict__ local,
                                                           u64* __restrict__ sums) {
    __shared__ uint8_t s_ntri[256];
    __shared__ u64 s_wave[kMeshThreads / 64];
    s_ntri[threadIdx.x] = T->ntri[threadIdx.x];
    __syncthreads();
    const u32 seg = blockIdx.x * kScanBlock + threadIdx.x;
    u64 tot = 0;
    if (seg < M.nseg) {
        const McWords W(M, seg);
        const u32 e = static_cast<u32>(__popcll(W.edges(0)) + __popcll(W.edges(1)) +
                                       __popcll(W.edges(2)));
        const u64 cubes = W.cubes();
        u32 t = 0;
        for (u64 m = cubes; m; m &= m - 1)
            t += s_ntri[W.config(static_cast<u32>(__ffsll(static_cast<unsigned long long>(m)) - 1))];
        tot = static_cast<u64>(e) | (static_cast<u64>(t) << kTriShift) |
              (static_cast<u64>(__popcll(cubes)) << kCubeShift);
    }
    const u32 lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    u64 x = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const u64 y = __shfl_up(x, o, 64);
        if (lane >= static_cast<u32>(o)) x += y;
    }
    if (lane == 63) s_wave[w] = x;
    __syncthreads();
    u64 run = x - tot;
    for (u32 k = 0; k < w; ++k) run += s_wave[k];
    if (seg < M.nseg) local[seg] = run;
    if (threadIdx.x == kMeshThreads - 1) sums[blockIdx.x] = run + tot;
}

// Exclusive scan of the block sums by one workgroup; totals: vertices and
// triangles.
constexpr int kSumThreads = 1024;
struct McBase {
    u32 verts, tris;
};
__global__ __launch_bounds__(kSumThreads) void k_mc_sums(const u64* __restrict__ sums, u32 nb,
                                                         McBase* __restrict__ base,
                                                         u64* __restrict__ totals) {
    __shared__ u64 s_wave[2][kSumThreads / 64];
    const u32 lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    u64 carry[2] = {0, 0};
    for (u32 b0 = 0; b0 < nb; b0 += kSumThreads) {
        const u32 b = b0 + threadIdx.x;
        const u64 v = b < nb ? sums[b] : 0ull;
        const u64 own[2] = {scan_verts(v), scan_tris(v)};
        u64 x[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            x[q] = own[q];
            for (int o = 1; o < 64; o <<= 1) {
                const u64 y = __shfl_up(x[q], o, 64);
                if (lane >= static_cast<u32>(o)) x[q] += y;
            }
            if (lane == 63) s_wave[q][w] = x[q];
        }
        __syncthreads();
        u64 off[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            off[q] = carry[q] + x[q] - own[q];
            for (u32 k = 0; k < kSumThreads / 64; ++k) {
                if (k < w) off[q] += s_wave[q][k];
                carry[q] += s_wave[q][k];
            }
        }
        if (b < nb) base[b] = McBase{static_cast<u32>(off[0]), static_cast<u32>(off[1])};
        __syncthreads();
    }
    if (threadIdx.x < 2) totals[threadIdx.x] = threadIdx.x == 0 ? carry[0] : carry[1];
}

// Index of the k-th set bit (k < popcount) of up to three masks read in bit
// order, mask after mask within a bit; also the mask it lies in.
__device__ __forceinline__ u32 nth_bit(u64 x, u64 y, u64 z, u32 k, u32& mask) {
    u32 at = 0;
#pragma unroll
    for (u32 step = 32; step > 0; step >>= 1) {
        const u64 low = (1ull << step) - 1ull;
        const u32 n = static_cast<u32>(__popcll((x >> at) & low) + __popcll((y >> at) & low) +
                                       __popcll((z >> at) & low));
        if (k >= n) {
            k -= n;
            at += step;
        }
    }
    const u32 bx = static_cast<u32>(x >> at) & 1u, by = static_cast<u32>(y >> at) & 1u;
    // k: number of set bits of the masks at `at` before the wanted one
    mask = (bx && k == 0) ? 0u : (by && k == bx) ? 1u : 2u;
    return at;
}
// Last entry of the ascending s[0..n) that is <= v (s[0] <= v).
__device__ __forceinline__ u32 last_at_most(const u32* s, u32 n, u32 v) {
    u32 lo = 0, hi = n - 1;
    while (lo < hi) {
        const u32 mid = (lo + hi + 1) >> 1;
        if (s[mid] <= v) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// Vertices, a workgroup per scan block and a thread per vertex: its segment by
// a search of the block's scan, its edge by the bits of the segment's words.
// Outputs of consecutive threads are consecutive (a wave per segment filled a
// few lanes and waited for one segment after the other: 211 us for 1.78
// million vertices).  Every grid point with crossing edges also records its
// edge mask and first vertex.  wide (with vpt): the binary64 copies that the
// smoothing starts from, instead of verts.
__global__ __launch_bounds__(kMeshThreads) void k_mc_vertices(
    const float* __restrict__ g, MeshGeom G, McGrid M, float iso, const u64* __restrict__ local,
    const u64* __restrict__ sums, const McBase* __restrict__ base, uint8_t* __restrict__ emask,
    u32* __restrict__ eoff, float* __restrict__ verts, double* __restrict__ wide,
    u32* __restrict__ vpt) {
    __shared__ u64 s_x[3][kScanBlock];
    __shared__ u32 s_first[kScanBlock];
    const u32 total = scan_verts(sums[blockIdx.x]);
    if (total == 0) return;
    const u32 seg0 = blockIdx.x * kScanBlock, seg = seg0 + threadIdx.x;
    const u32 nseg = min(static_cast<u32>(kScanBlock), M.nseg - seg0);
    if (threadIdx.x < nseg) {
        const McWords W(M, seg);
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) s_x[ax][threadIdx.x] = W.edges(ax);
        s_first[threadIdx.x] = scan_verts(local[seg]);
    }
    __syncthreads();
    const u64 v0 = base[blockIdx.x].verts;
    const u64 st[3] = {static_cast<u64>(M.r1) * M.r2, static_cast<u64>(M.r2), 1};
    const double lo[3] = {G.lo0, G.lo1, G.lo2}, sp[3] = {G.sp0, G.sp1, G.sp2};
    for (u32 k = threadIdx.x; k < total; k += kMeshThreads) {
        const u32 t = last_at_most(s_first, nseg, k);
        const u64 xa = s_x[0][t], xb = s_x[1][t], xc = s_x[2][t];
        u32 ax;
        const u32 bit = nth_bit(xa, xb, xc, k - s_first[t], ax);
        const u32 row = (seg0 + t) / M.ntx;
        const u32 a = row / static_cast<u32>(M.r1), b = row - a * static_cast<u32>(M.r1);
        const u32 c = (seg0 + t - row * M.ntx) * 64u + bit;
        const u64 i = static_cast<u64>(row) * M.r2 + c;
        const double g0 = static_cast<double>(g[i]);
        const double g1 = static_cast<double>(g[i + (ax == 0 ? st[0] : ax == 1 ? st[1] : st[2])]);
        const u32 m = (static_cast<u32>(xa >> bit) & 1u) | ((static_cast<u32>(xb >> bit) & 1u) << 1) |
                      ((static_cast<u32>(xc >> bit) & 1u) << 2);
        const u64 v = v0 + k;
        if ((m & ((1u << ax) - 1u)) == 0u) {  // the point's first vertex
            emask[i] = static_cast<uint8_t>(m);
            eoff[i] = static_cast<u32>(v);
        }
        const double f = (static_cast<double>(iso) - g0) / (g1 - g0);
        const u32 idx[3] = {a, b, c};
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const double at = static_cast<double>(static_cast<int>(idx[q]));
            const double w = static_cast<u32>(q) == ax ? at + f : at;
            const float p = static_cast<float>(w * sp[q] + lo[q]);
            if (wide) wide[3 * v + q] = static_cast<double>(p);
            else verts[3 * v + q] = p;
        }
        if (vpt) vpt[v] = static_cast<u32>(i) << 2 | ax;
    }
}

// Offsets of a cube edge's owner corner and the edge's axis: bit ax clear, the
// other two bits from the edge id (lower axis first).
__device__ __forceinline__ u64 edge_owner(u64 cube, int e, u64 sa, u64 sb, int& ax) {
    ax = e >> 2;
    const int b0 = e & 1, b1 = (e >> 1) & 1;
    const int oa = ax == 0 ? 0 : b0;
    const int ob = ax == 0 ? b0 : ax == 1 ? 0 : b1;
    const int oc = ax == 2 ? 0 : b1;
    return cube + (oa ? sa : 0ull) + (ob ? sb : 0ull) + static_cast<u64>(oc);
}

// Triangles, a workgroup per scan block and a thread per cube that has any:
// cubes in order, a chunk of kMeshThreads at a time, their places from a scan
// of the chunk's triangle counts (a wave per segment: 341 us for 3.54 million
// triangles).  Every vertex is the owner grid point's first vertex plus the
// crossing edges it owns on lower axes.
__global__ __launch_bounds__(kMeshThreads) void k_mc_triangles(
    McGrid M, const McDev* __restrict__ T, const u64* __restrict__ local,
    const u64* __restrict__ sums, const McBase* __restrict__ base,
    const uint8_t* __restrict__ emask, const u32* __restrict__ eoff, u32* __restrict__ tris) {
    __shared__ __align__(16) McDev sT;
    __shared__ u64 s_act[kScanBlock];
    __shared__ u32 s_first[kScanBlock];
    __shared__ u32 s_wave[kMeshThreads / 64];
    const u32 total = scan_cubes(sums[blockIdx.x]);
    if (total == 0) return;
    for (u32 k = threadIdx.x; k < sizeof(McDev) / 4; k += kMeshThreads)
        reinterpret_cast<u32*>(&sT)[k] = reinterpret_cast<const u32*>(T)[k];
    const u32 seg0 = blockIdx.x * kScanBlock;
    const u32 nseg = min(static_cast<u32>(kScanBlock), M.nseg - seg0);
    if (threadIdx.x < nseg) {
        const McWords W(M, seg0 + threadIdx.x);
        s_act[threadIdx.x] = W.cubes();
        s_first[threadIdx.x] = scan_cubes(local[seg0 + threadIdx.x]);
    }
    __syncthreads();
    const u64 sa = static_cast<u64>(M.r1) * M.r2, sb = static_cast<u64>(M.r2);
    const u32 lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    u64 t0 = base[blockIdx.x].tris;
    for (u32 k0 = 0; k0 < total; k0 += kMeshThreads) {
        const u32 k = k0 + threadIdx.x;
        u32 cfg = 0, nt = 0;
        u64 i = 0;
        if (k < total) {
            const u32 t = last_at_most(s_first, nseg, k);
            u32 unused;
            const u32 bit = nth_bit(s_act[t], 0ull, 0ull, k - s_first[t], unused);
            const McWords W(M, seg0 + t);
            cfg = W.config(bit);
            nt = sT.ntri[cfg];
            i = (static_cast<u64>(W.a) * M.r1 + W.b) * M.r2 + W.tx * 64u + bit;
        }
        u32 x = nt;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const u32 y = __shfl_up(x, o, 64);
            if (lane >= static_cast<u32>(o)) x += y;
        }
        if (lane == 63) s_wave[w] = x;
        __syncthreads();
        u64 at = t0 + x - nt;
        for (u32 q = 0; q < kMeshThreads / 64; ++q) {
            if (q < w) at += s_wave[q];
            t0 += s_wave[q];
        }
        __syncthreads();
        for (u32 t = 0; t < nt; ++t) {
            u32 out[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                int ax;
                const u64 o = edge_owner(i, sT.tri[cfg][3 * t + q], sa, sb, ax);
                out[q] = eoff[o] + static_cast<u32>(__popc(emask[o] & ((1u << ax) - 1u)));
            }
#pragma unroll
            for (int q = 0; q < 3; ++q) tris[3 * (at + t) + q] = out[q];
        }
    }
}

// ---- Laplacian mesh smoothing ---------------------------------------------
// Open3D's TriangleMesh::filter_smooth_laplacian (the reference's
// mesh.filter_smooth_laplacian(number_of_iterations=n), default lambda 0.5),
// as its documentation states it: every vertex moves to
// v + lambda (sum_n w_n v_n / sum_n w_n - v), w_n = 1 / (|v - v_n| + 1e-12),
// over the vertices that share a triangle with it, all from the previous
// pass, in binary64.  The sums here run over the neighbours in ascending
// index (Open3D's hash-set order is unspecified).
// Neighbours per vertex: a cube's table has at most 5 triangles, so a vertex
// sits on one fan of at most 7 vertices per cube and has at most 6
// neighbours there, 24 over the four cubes around its edge.
constexpr int kAdjCap = 24;

// Neighbours of the vertex on grid edge (i, ax), in ascending order, from the
// (up to) four cubes around the edge: the other vertices of the table
// triangles that contain it.  Returns their number, or CAP + 1 if there are
// more than CAP.
template <int CAP>
__device__ __forceinline__ u32 mc_neighbours(const McGrid& M, const McDev& T, u32 i32, int ax,
                                             const uint8_t* __restrict__ emask,
                                             const u32* __restrict__ eoff, u32 (&L)[CAP]) {
    const u32 plane = static_cast<u32>(M.r1) * static_cast<u32>(M.r2);
    const int a = static_cast<int>(i32 / plane), rem = static_cast<int>(i32 % plane);
    const int idx[3] = {a, rem / M.r2, rem % M.r2};
    const int r[3] = {M.r0, M.r1, M.r2};
    const u64 st[3] = {plane, static_cast<u64>(M.r2), 1};
    // inside bits of points c and c + 1 of row (a, b)
    auto two = [&](int ra, int rb, int c) -> u32 {
        const u32 t = (static_cast<u32>(ra) * M.r1 + rb) * M.ntx + (static_cast<u32>(c) >> 6);
        const u32 k = static_cast<u32>(c) & 63u;
        if (k < 63u) return static_cast<u32>(M.bits[t] >> k) & 3u;
        return static_cast<u32>(M.bits[t] >> 63) | (static_cast<u32>(M.bits[t + 1] & 1ull) << 1);
    };
#pragma unroll
    for (int k = 0; k < CAP; ++k) L[k] = 0xFFFFFFFFu;
    u32 n = 0;
    const int u = ax == 0 ? 1 : 0, w = ax == 2 ? 1 : 2;  // the other axes, lower first
    for (int o = 0; o < 4; ++o) {
        const int ou = o & 1, ow = o >> 1;
        // the cube whose lowest corner is this point - ou e_u - ow e_w
        int q0[3] = {idx[0], idx[1], idx[2]};
        q0[u] -= ou;
        q0[w] -= ow;
        if (q0[u] < 0 || q0[w] < 0 || q0[u] + 1 >= r[u] || q0[w] + 1 >= r[w]) continue;
        const u64 qi = static_cast<u64>(i32) - ou * st[u] - ow * st[w];
        u32 cfg = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const u32 c2 = two(q0[0] + (k & 1), q0[1] + (k >> 1), q0[2]);
            cfg |= ((c2 & 1u) << k) | ((c2 >> 1) << (k + 4));
        }
        const int mine = 4 * ax + (ou | (ow << 1));  // this edge within that cube
        for (u32 t = 0; t < T.ntri[cfg]; ++t) {
            const uint8_t* tri = T.tri[cfg] + 3 * t;
            if (tri[0] != mine && tri[1] != mine && tri[2] != mine) continue;
            for (int q = 0; q < 3; ++q) {
                const int e = tri[q];
                if (e == mine) continue;
                int eax;
                const u64 oi = edge_owner(qi, e, st[0], st[1], eax);
                u32 y = eoff[oi] + static_cast<u32>(__popc(emask[oi] & ((1u << eax) - 1u)));
                bool seen = false;
#pragma unroll
                for (int k2 = 0; k2 < CAP; ++k2) seen |= L[k2] == y;
                if (seen) continue;
                if (n == static_cast<u32>(CAP)) return CAP + 1;
#pragma unroll
                for (int k2 = 0; k2 < CAP; ++k2) {  // sorted insert
                    const bool less = y < L[k2];
                    const u32 tk = L[k2];
                    L[k2] = less ? y : tk;
                    y = less ? tk : y;
                }
                ++n;
            }
        }
    }
    return n;
}

// Neighbours of every vertex, a thread each: in a short register list first (a
// vertex has about six, and every insertion passes the whole list), in the
// full one for the vertices with more.  Those are few on smooth surfaces, and
// kAdjAll takes them on the spot.  On rugged ones they make nearly every wave
// go through both lists, so from kAdjSplit vertices on kAdjFirst lists them for
// a launch of their own, kAdjRest (18.5 million vertices of a splash: 4,209 ->
// 3,300 us; below, the launch costs what it saves).
constexpr int kAdjShort = 9;
constexpr u64 kAdjSplit = 262144;
enum { kAdjAll, kAdjFirst, kAdjRest };
template <int CAP>
__device__ __forceinline__ void adj_store(u32* __restrict__ row, const u32 (&L)[CAP], u32 n) {
#pragma unroll
    for (int k = 0; k < CAP; ++k)
        if (static_cast<u32>(k) < n) row[k] = L[k];
}
template <int MODE>
__global__ __launch_bounds__(256) void k_mc_adjacency(McGrid M, const McDev* __restrict__ T,
                                                      u64 nvert, const u32* __restrict__ vpt,
                                                      const uint8_t* __restrict__ emask,
                                                      const u32* __restrict__ eoff,
                                                      u32* __restrict__ adj,
                                                      u32* __restrict__ deg, SplitList more,
                                                      u32* __restrict__ over) {
    __shared__ __align__(16) McDev sT;  // the table, read per lane below
    for (u32 k = threadIdx.x; k < sizeof(McDev) / 4; k += 256)
        reinterpret_cast<u32*>(&sT)[k] = reinterpret_cast<const u32*>(T)[k];
    __syncthreads();
    constexpr bool kRest = MODE == kAdjRest;
    // an XCD takes a run of vertices: neighbours lie within a few planes, in its L2
    const u32 part = blockIdx.x % kParts;
    const u32 b = kRest ? blockIdx.x / kParts : xcd_tile(blockIdx.x, gridDim.x);
    const u64 count = kRest ? static_cast<u64>(more.size(part)) : nvert;
    const u64 stride = static_cast<u64>(kRest ? gridDim.x / kParts : gridDim.x) * 256;
    for (u64 t = static_cast<u64>(b) * 256 + threadIdx.x; t < count; t += stride) {
        const u32 v = kRest ? more.at(part, static_cast<u32>(t)) : static_cast<u32>(t);
        const u32 code = vpt[v];  // its grid edge: from grid point i (< 2^30) along an axis
        const int ax = static_cast<int>(code & 3u);
        u32* row = adj + static_cast<u64>(v) * kAdjCap;
        u32 n = kAdjShort + 1;
        if constexpr (!kRest) {
            u32 L[kAdjShort];
            n = mc_neighbours<kAdjShort>(M, sT, code >> 2, ax, emask, eoff, L);
            if (n <= static_cast<u32>(kAdjShort)) adj_store(row, L, n);
        }
        if (n > static_cast<u32>(kAdjShort)) {
            if constexpr (MODE == kAdjFirst) {
                more.wave_append(part, v);
                continue;
            } else {
                u32 F[kAdjCap];
                n = mc_neighbours<kAdjCap>(M, sT, code >> 2, ax, emask, eoff, F);
                if (n > static_cast<u32>(kAdjCap)) {
                    atomicOr(over, 1u);
                    n = kAdjCap;
                }
                adj_store(row, F, n);
            }
        }
        deg[v] = n;
    }
}

__global__ __launch_bounds__(kMeshThreads) void k_verts_narrow(const double* __restrict__ in,
                                                               u64 n, float* __restrict__ out) {
    const u64 i = static_cast<u64>(blockIdx.x) * kMeshThreads + threadIdx.x;
    if (i < n) out[i] = static_cast<float>(in[i]);
}

__global__ __launch_bounds__(kMeshThreads) void k_mesh_laplacian(const double* __restrict__ V,
                                                                 u64 nv,
                                                                 const u32* __restrict__ adj,
                                                                 const u32* __restrict__ deg,
                                                                 double* __restrict__ out) {
    const u64 v = static_cast<u64>(xcd_tile(blockIdx.x, gridDim.x)) * kMeshThreads + threadIdx.x;
    if (v >= nv) return;
    const double px = V[3 * v], py = V[3 * v + 1], pz = V[3 * v + 2];
    double sx = 0.0, sy = 0.0, sz = 0.0, tw = 0.0;
    const u32* L = adj + v * kAdjCap;
    const u32 n = deg[v];
    for (u32 k = 0; k < n; ++k) {
        const u64 j = L[k];
        const double qx = V[3 * j], qy = V[3 * j + 1], qz = V[3 * j + 2];
        const double dx = px - qx, dy = py - qy, dz = pz - qz;
        const double wgt = 1.0 / (sqrt(dx * dx + dy * dy + dz * dz) + 1e-12);
        tw = tw + wgt;
        sx = sx + wgt * qx;
        sy = sy + wgt * qy;
        sz = sz + wgt * qz;
    }
    out[3 * v] = px + 0.5 * (sx / tw - px);
    out[3 * v + 1] = py + 0.5 * (sy / tw - py);
    out[3 * v + 2] = pz + 0.5 * (sz / tw - pz);
}

}  // namespace

// numpy's float64 sum: sequential below 8 elements, eight running sums
// combined pairwise up to 128, halves (a multiple of 8 first) beyond.
static double numpy_sum(const double* a, size_t n) {
    if (n < 8) {
        double r = 0.0;
        for (size_t i = 0; i < n; ++i) r = r + a[i];
        return r;
    }
    if (n <= 128) {
        double r[8];
        for (int j = 0; j < 8; ++j) r[j] = a[j];
        size_t i = 8;
        for (; i < n - n % 8; i += 8)
            for (int j = 0; j < 8; ++j) r[j] = r[j] + a[i + j];
        double res = ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
        for (; i < n; ++i) res = res + a[i];
        return res;
    }
    size_t n2 = n / 2;
    n2 -= n2 % 8;
    return numpy_sum(a, n2) + numpy_sum(a + n2, n - n2);
}

// One smoothing pass over the gridded points: the guessed radius in rings 0..1,
// then the points it held too many or too few neighbours for (surfaces, other
// spacings; rings 0..4 reach k points at four times the expected spacing),
// then dense and far neighbourhoods.
constexpr u32 kNearLanes = 8;  // lanes per point of the first searches
constexpr u32 kNearPoints = kMeshThreads / kNearLanes;
template <int K>
static void knn_pass(const double* in, u32 n, const KnnGrid& kg, const u32* sorted,
                     const double* ps, const u32* cs, double* out, u32* counts, u32* lists,
                     hipStream_t s) {
    constexpr u32 kWideLanes = 16, kWaveLanes = 64;
    const u32 tiles = div_up(n, kNearPoints), cap = part_capacity(tiles, kNearPoints);
    auto list = [&](u32 k) {
        return SplitList{counts + k * kPartCounts, lists + static_cast<u64>(k) * kParts * cap, cap};
    };
    static_assert(kKnnLists == 5, "one each");
    const SplitList few = list(0), many = list(1), fewer = list(2), rest = list(3), far = list(4);
    // (a launch holds fewer than 2^32 threads, eight a point here: 2^29 points;
    // the groups stride over what is left)
    constexpr u32 kGroupBlocks = 1u << 16;
    // workgroups of a list's consumer: the same number for every part
    auto blocks = [&](u32 per, u32 most) {
        return std::min(div_up(div_up(n, per), kParts) * kParts, most);
    };
    k_knn_group<K, 1, kNearLanes, true><<<std::min(tiles, kGroupBlocks), kMeshThreads, 0, s>>>(
        n, SplitList{}, kg, sorted, ps, cs, out, few, many);
    WSIM_LAUNCH_CHECK();
    k_knn_group<K, 1, kNearLanes, false><<<blocks(kNearPoints, 2048), kMeshThreads, 0, s>>>(
        n, many, kg, sorted, ps, cs, out, few, rest);
    WSIM_LAUNCH_CHECK();
    k_knn_group<K, 2, kWideLanes, false>
        <<<blocks(kMeshThreads / kWideLanes, 2048), kMeshThreads, 0, s>>>(
            n, few, kg, sorted, ps, cs, out, fewer, rest);
    WSIM_LAUNCH_CHECK();
    k_knn_group<K, 4, kWaveLanes, false>
        <<<blocks(kMeshThreads / kWaveLanes, 2048), kMeshThreads, 0, s>>>(
            n, fewer, kg, sorted, ps, cs, out, rest, rest);
    WSIM_LAUNCH_CHECK();
    k_knn_smooth<K><<<blocks(kMeshThreads, 1024), kMeshThreads, 0, s>>>(in, kg, sorted, ps, cs,
                                                                        rest, out, far);
    WSIM_LAUNCH_CHECK();
    // 4 waves per workgroup walk the list
    k_knn_far<K><<<blocks(kMeshThreads, 256), kMeshThreads, 0, s>>>(in, kg, sorted, ps, cs, far, out);
    WSIM_LAUNCH_CHECK();
}

// Radius of a sphere that holds k points at one per unit volume.
static double knn_radius(double k) {
    return std::cbrt(k * 3.0 / (4.0 * 3.14159265358979));
}

std::vector<double> gaussian_weights(double sigma, int* radius) {
    // scipy.ndimage._gaussian_kernel1d, order 0, truncate 4.0: phi / phi.sum()
    const int R = static_cast<int>(4.0 * sigma + 0.5);
    std::vector<double> w(2 * R + 1);
    const double s2 = sigma * sigma;
    for (int k = -R; k <= R; ++k) {
        w[k + R] = std::exp(-0.5 / s2 * static_cast<double>(k * k));
    }
    const double sum = numpy_sum(w.data(), w.size());
    for (double& x : w) x = x / sum;
    *radius = R;
    return w;
}

const uint8_t* mc_table_counts() { return mc_table().ntri; }
const uint8_t* mc_table_triangles() { return &mc_table().tri[0][0]; }

SurfaceMesher::SurfaceMesher(hipStream_t stream) : stream_(stream) {}

void SurfaceMesher::run(const float* xyz, size_t n, const MeshParams& P) {
    if (!xyz && n) fail(kInvalidArgument, "SurfaceMesher: NULL positions");
    if (n == 0) fail(kInvalidArgument, "SurfaceMesher: no points");
    if (!(P.particle_radius > 0.0) || !(P.grid_voxel_factor > 0.0) || !(P.smooth_sigma >= 0.0))
        fail(kInvalidArgument, "SurfaceMesher: radius, voxel factor and sigma must be positive");
    if (P.smooth_pre_iters < 0 || P.smooth_post_iters < 0)
        fail(kInvalidArgument, "SurfaceMesher: negative smoothing iterations");
    if (P.smooth_pre_iters > 0) {
        const int k = P.k_neighbors;
        if (k != 8 && k != 10 && k != 15 && k != 20 && k != 30)
            fail(kInvalidArgument, "SurfaceMesher: k_neighbors must be 8, 10, 15, 20 or 30");
        if (n < static_cast<size_t>(k))
            fail(kInvalidArgument, "SurfaceMesher: fewer points than k_neighbors");
    }
    if (n > 0xFFFFF000ull) fail(kInvalidArgument, "SurfaceMesher: too many points");
    hipStream_t s = stream_;
    const u32 nn = static_cast<u32>(n);
    const u32 gp = div_up(nn, static_cast<u32>(kMeshThreads));
    if (pts_[0].size() < 3 * n) {
        pts_[0] = DeviceBuffer<double>(3 * n);
        pts_[1] = DeviceBuffer<double>(3 * n);
    }
    k_mesh_points<<<gp, kMeshThreads, 0, s>>>(xyz, n, P.swap_yz ? 1 : 0, pts_[0].data());
    WSIM_LAUNCH_CHECK();
    // small results are read through one pinned buffer, and the small device
    // buffers stay allocated between runs (an allocation or a free waits for
    // the device)
    auto fit = [](auto& b, u64 want) {
        if (b.size() < want) b = std::remove_reference_t<decltype(b)>(want);
    };
    constexpr u32 kBoundsBlocks = 256;
    const u32 nbb = std::min<u32>(gp, kBoundsBlocks);
    fit(bpart_, kBoundsPart * static_cast<u64>(kBoundsBlocks));
    fit(hostbuf_, kBoundsPart * static_cast<u64>(kBoundsBlocks));
    auto read_back = [&](void* dst, const void* src, size_t bytes) {
        WSIM_HIP(hipMemcpyAsync(hostbuf_.data(), src, bytes, hipMemcpyDeviceToHost, s));
        WSIM_HIP(hipStreamSynchronize(s));
        std::memcpy(dst, hostbuf_.data(), bytes);
    };
    auto bounds = [&](const double* pts, double* mn, double* mx) {
        k_mesh_bounds<<<nbb, kMeshThreads, 0, s>>>(pts, n, bpart_.data());
        WSIM_LAUNCH_CHECK();
        double hp[kBoundsPart * kBoundsBlocks];
        read_back(hp, bpart_.data(), kBoundsPart * static_cast<size_t>(nbb) * sizeof(double));
        for (int a = 0; a < 3; ++a) {
            mn[a] = INFINITY;
            mx[a] = -INFINITY;
        }
        double bad = 0.0;
        for (u32 k = 0; k < nbb; ++k) {
            for (int a = 0; a < 3; ++a) {
                mn[a] = std::fmin(mn[a], hp[kBoundsPart * k + a]);
                mx[a] = std::fmax(mx[a], hp[kBoundsPart * k + 3 + a]);
            }
            bad += hp[kBoundsPart * k + 6];
        }
        if (bad != 0.0) fail(kInvalidArgument, "SurfaceMesher: non-finite positions");
        for (int a = 0; a < 3; ++a)
            if (!std::isfinite(mn[a]) || !std::isfinite(mx[a]))
                fail(kInvalidArgument, "SurfaceMesher: non-finite positions");
    };
    // 1. k-nearest-neighbour position smoothing (:61-74)
    int cur = 0;
    double mn[3], mx[3];
    double dia = 2.0 * P.particle_radius;  // expected spacing
    for (int it = 0; it < P.smooth_pre_iters; ++it) {
        bounds(pts_[cur].data(), mn, mx);
        KnnGrid kg{};
        kg.lo0 = mn[0], kg.lo1 = mn[1], kg.lo2 = mn[2];
        // The spacing: a particle diameter, or less where the points' box
        // holds more of them.  The guess holds about k + 4 points at it, and
        // a cell's edge is the guess, so rings 0..1 reach it (a pass of
        // 1,001,385 points: 312 us; 353 with cells 1.15 times as wide; with
        // 0.85 most points fall short and take 1,400).
        const double box = (mx[0] - mn[0] + dia) * (mx[1] - mn[1] + dia) * (mx[2] - mn[2] + dia);
        const double room = std::cbrt(box / static_cast<double>(n));
        const double unit = knn_radius(P.k_neighbors + 4.0);
        double gr = unit * std::min(dia, room);
        kg.cell = gr;
        if (knn_keys_[0].size() < n) {
            for (auto& b : knn_keys_) b = DeviceBuffer<u32>(n);
            for (auto& b : knn_vals_) b = DeviceBuffer<u32>(n);
            knn_hist_ = DeviceBuffer<u32>(radix_hist_elems(n));
        }
        fit(knn_farc_, kKnnLists * kPartCounts);
        int w = 0;
        auto sort_cells = [&] {
            u64 cells = 0;
            for (;;) {
                kg.d0 = static_cast<int>((mx[0] - mn[0]) / kg.cell) + 1;
                kg.d1 = static_cast<int>((mx[1] - mn[1]) / kg.cell) + 1;
                kg.d2 = static_cast<int>((mx[2] - mn[2]) / kg.cell) + 1;
                cells = static_cast<u64>(kg.d0) * kg.d1 * kg.d2;
                if (cells <= (1ull << 26)) break;
                kg.cell *= 2.0;
            }
            k_knn_keys<<<gp, kMeshThreads, 0, s>>>(pts_[cur].data(), nn, kg, knn_keys_[0].data(),
                                                   knn_vals_[0].data());
            WSIM_LAUNCH_CHECK();
            w = radix_sort_pairs(knn_keys_[0].data(), knn_vals_[0].data(), knn_keys_[1].data(),
                                 knn_vals_[1].data(), n, key_bits(static_cast<u32>(cells - 1)),
                                 knn_hist_.data(), s);
            return cells;
        };
        u64 cells = sort_cells();
        // A box with room for ten times the points at that spacing is one of
        // spray, or the radius is well below the spacing: then nearly every
        // point would fall short of the guess and go through all the wide
        // searches.  A cell that holds little more than a point tells, and
        // doubled cells until they hold as many as the guess does give the
        // spacing, once a run.  Two passes over 97,290 points, us: radius 3
        // times too small 2,104 -> 499, 10 times 20,519 -> 598 (right: 340;
        // 17,550 points, half the radius: 312 -> 382, the price of the waits).
        if (it == 0 && room > 2.2 * dia) {
            auto points_per_cell = [&] {
                u32 used = 0;
                WSIM_HIP(hipMemsetAsync(knn_farc_.data(), 0, sizeof(u32), s));
                k_knn_used<<<std::min<u32>(gp, 256), kMeshThreads, 0, s>>>(knn_keys_[w].data(), nn,
                                                                           knn_farc_.data());
                WSIM_LAUNCH_CHECK();
                read_back(&used, knn_farc_.data(), sizeof(u32));
                return static_cast<double>(n) / static_cast<double>(used);
            };
            double held = points_per_cell();
            if (held < 1.3) {
                while (cells > 1 && held < unit * unit * unit) {
                    kg.cell *= 2.0;
                    cells = sort_cells();
                    held = points_per_cell();
                }
                dia = kg.cell / std::cbrt(held);
                gr = unit * dia;
                kg.cell = gr;
                cells = sort_cells();
            }
        }
        kg.guess = gr * gr;
        if (knn_cs_.size() < cells + 1) knn_cs_ = DeviceBuffer<u32>(cells + 1);
        build_cell_start(knn_keys_[w].data(), nn, static_cast<u32>(cells + 1), knn_cs_.data(), s,
                         0);
        const u32* sorted = knn_vals_[w].data();
        double* out = pts_[cur ^ 1].data();
        if (knn_ps_.size() < 3 * n) knn_ps_ = DeviceBuffer<double>(3 * n);
        k_knn_gather<<<gp, kMeshThreads, 0, s>>>(pts_[cur].data(), nn, sorted, knn_ps_.data());
        WSIM_LAUNCH_CHECK();
        const double* in = pts_[cur].data();
        const double* ps = knn_ps_.data();
        const u32* cs = knn_cs_.data();
        fit(knn_far_, static_cast<u64>(kKnnLists) * kParts *
                          part_capacity(div_up(n, kNearPoints), kNearPoints));
        u32* fc = knn_farc_.data();  // counts of the lists
        WSIM_HIP(hipMemsetAsync(fc, 0, kKnnLists * kPartCounts * sizeof(u32), s));
        u32* lists = knn_far_.data();
        switch (P.k_neighbors) {
        case 8: knn_pass<8>(in, nn, kg, sorted, ps, cs, out, fc, lists, s); break;
        case 10: knn_pass<10>(in, nn, kg, sorted, ps, cs, out, fc, lists, s); break;
        case 15: knn_pass<15>(in, nn, kg, sorted, ps, cs, out, fc, lists, s); break;
        case 20: knn_pass<20>(in, nn, kg, sorted, ps, cs, out, fc, lists, s); break;
        default: knn_pass<30>(in, nn, kg, sorted, ps, cs, out, fc, lists, s); break;
        }
        cur ^= 1;
    }
    const double* pts = pts_[cur].data();
    bounds(pts, mn, mx);
    // 2. grid (tools/particles_to_mesh.py:104-109), binary64 as numpy
    const double pad = P.particle_radius * 4.0;
    const double voxel = P.particle_radius * P.grid_voxel_factor;
    MeshGeom G{};
    int res[3];
    double lo[3], ext[3];
    for (int a = 0; a < 3; ++a) {
        lo[a] = mn[a] - pad;
        const double hi = mx[a] + pad;
        ext[a] = hi - lo[a];
        const double r = std::ceil(ext[a] / voxel);
        if (!(r < 65536.0)) fail(kOutOfRange, "SurfaceMesher: grid too large");
        res[a] = std::max(static_cast<int>(r), 8);
    }
    G.r0 = res[0], G.r1 = res[1], G.r2 = res[2];
    G.lo0 = lo[0], G.lo1 = lo[1], G.lo2 = lo[2];
    G.ext0 = ext[0], G.ext1 = ext[1], G.ext2 = ext[2];
    G.sp0 = ext[0] / res[0], G.sp1 = ext[1] / res[1], G.sp2 = ext[2] / res[2];
    const u64 nv = static_cast<u64>(res[0]) * res[1] * res[2];
    if (nv > (1ull << 31)) fail(kOutOfRange, "SurfaceMesher: grid too large");
    info_ = MeshInfo{};
    for (int a = 0; a < 3; ++a) {
        info_.dims[a] = res[a];
        info_.lo[a] = lo[a];
        info_.extent[a] = ext[a];
    }
    info_.spacing[0] = G.sp0, info_.spacing[1] = G.sp1, info_.spacing[2] = G.sp2;
    const u32 gv = static_cast<u32>((nv + kMeshThreads - 1) / kMeshThreads);
    // grid-sized work buffers are kept between runs and grow as needed
    fit(grid_, nv);
    fit(tmp_, nv);
    fit(count_, nv);
    fit(eoff_, nv);
    fit(emask_, nv);
    // 3. splat
    u32* count = count_.data();
    WSIM_HIP(hipMemsetAsync(count, 0, nv * sizeof(u32), s));
    k_mesh_splat<<<gp, kMeshThreads, 0, s>>>(pts, n, G, count);
    WSIM_LAUNCH_CHECK();
    // 4. blur and 5. the maximum for the iso level
    int R = 0;
    std::vector<double> w;
    if (P.smooth_sigma > 0.0) {
        w = gaussian_weights(P.smooth_sigma, &R);
        if (P.weights) std::memcpy(w.data(), P.weights, w.size() * sizeof(double));
        if (R <= 16) {  // the compile-time radii of the tiled passes (0 weights change no sum)
            const size_t pad = static_cast<size_t>((R <= 10 ? 10 : 16) - R);
            w.insert(w.begin(), pad, 0.0);
            w.insert(w.end(), pad, 0.0);
        }
        fit(weights_, w.size());
        WSIM_HIP(hipMemcpyAsync(weights_.data(), w.data(), w.size() * sizeof(double),
                                hipMemcpyHostToDevice, s));
    }
    auto max_of = [&](const float* a, u64 na) {
        constexpr u32 kMaxBlocks = 1024;
        static_assert(kMaxBlocks * sizeof(float) <= kBoundsPart * kBoundsBlocks * sizeof(double),
                      "read through hostbuf_");
        const u32 nbm = static_cast<u32>(
            std::min<u64>((na + kMeshThreads - 1) / kMeshThreads, kMaxBlocks));
        fit(mpart_, kMaxBlocks);
        k_mesh_max<<<nbm, kMeshThreads, 0, s>>>(a, na, mpart_.data());
        WSIM_LAUNCH_CHECK();
        float hm[kMaxBlocks];
        read_back(hm, mpart_.data(), nbm * sizeof(float));
        float m = -INFINITY;
        for (u32 k = 0; k < nbm; ++k) m = std::fmax(m, hm[k]);
        return m;
    };
    float gmax;
    if (P.smooth_sigma > 0.0 && R <= kBlurMaxR) {
        // counts -> grid_ (axis 0) -> tmp_ (axis 1) -> grid_ (axis 2), with
        // compile-time radii up to 16 (weights padded with zeros)
        const int RT = R <= 10 ? 10 : R <= 16 ? 16 : R;
        const u32 area = static_cast<u32>(res[1]) * static_cast<u32>(res[2]);
        const dim3 g0((area + 63) / 64, static_cast<u32>((res[0] + kBlurTile - 1) / kBlurTile), 1);
        const dim3 g1(static_cast<u32>((res[2] + 63) / 64),
                      static_cast<u32>((res[1] + kBlurTile - 1) / kBlurTile), static_cast<u32>(res[0]));
        const u64 rows = static_cast<u64>(res[0]) * res[1];
        const u64 nparts = (rows + 4 * kBlurRows - 1) / (4 * kBlurRows);
        fit(part_, nparts);
        auto blur = [&](auto rt) {
            constexpr int T = decltype(rt)::value;
            const size_t lds = static_cast<size_t>(kBlurTile + 2 * RT) * 64 * sizeof(float);
            k_blur_strided<u32, T><<<g0, 256, lds, s>>>(count, grid_.data(), area, res[0], nv,
                                                        weights_.data(), RT);
            WSIM_LAUNCH_CHECK();
            k_blur_strided<float, T><<<g1, 256, lds, s>>>(grid_.data(), tmp_.data(),
                                                          static_cast<u32>(res[2]), res[1], area,
                                                          weights_.data(), RT);
            WSIM_LAUNCH_CHECK();
            k_blur_rows<T><<<static_cast<u32>(nparts), 256,
                             4 * blur_row_floats(RT) * sizeof(float), s>>>(
                tmp_.data(), grid_.data(), rows, res[2], weights_.data(), RT, part_.data());
            WSIM_LAUNCH_CHECK();
        };
        if (RT == 10) blur(std::integral_constant<int, 10>{});
        else if (RT == 16) blur(std::integral_constant<int, 16>{});
        else blur(std::integral_constant<int, 0>{});
        gmax = max_of(part_.data(), nparts);
    } else {
        k_mesh_to_float<<<gv, kMeshThreads, 0, s>>>(count, grid_.data(), nv);
        WSIM_LAUNCH_CHECK();
        if (P.smooth_sigma > 0.0) {  // taps beyond the tiles' LDS: one load per tap
            float* src = grid_.data();
            float* dst = tmp_.data();
            for (int axis = 0; axis < 3; ++axis) {
                k_mesh_blur<<<gv, kMeshThreads, 0, s>>>(src, dst, res[0], res[1], res[2], axis,
                                                        weights_.data(), R);
                WSIM_LAUNCH_CHECK();
                std::swap(src, dst);
            }
            if (src != grid_.data()) std::swap(grid_, tmp_);
        }
        gmax = max_of(grid_.data(), nv);
    }
    info_.max_density = gmax;
    // numpy 2: float32 scalar * Python float stays float32
    const float iso = gmax * static_cast<float>(P.iso_factor);
    info_.iso = iso;
    info_.n_vertices = info_.n_triangles = 0;
    if (!(gmax > 0.0f)) return;
    // 6. marching cubes
    const McTable& T = mc_table();
    static_assert(sizeof(McDev) == sizeof(McTable), "table layout");
    if (table_.size() == 0) {  // uploaded once
        DeviceBuffer<uint8_t> t(sizeof(McTable));
        WSIM_HIP(hipMemcpyAsync(t.data(), &T, sizeof(McTable), hipMemcpyHostToDevice, s));
        table_ = std::move(t);
    }
    const McDev* dT = reinterpret_cast<const McDev*>(table_.data());
    const u32 ntx = static_cast<u32>((res[2] + 63) / 64);
    const u64 rows = static_cast<u64>(res[0]) * res[1];
    const u64 nseg = rows * ntx;  // < 2^31: at most one per voxel
    const u32 nb = static_cast<u32>((nseg + kScanBlock - 1) / kScanBlock);
    fit(bits_, nseg + 1);
    fit(local_, nseg);
    fit(sums_, nb);
    fit(base_, 2ull * nb);
    fit(totals_, 2);
    auto* base = reinterpret_cast<McBase*>(base_.data());
    const u32 gb = static_cast<u32>(std::min<u64>((nseg + 31) / 32, 8192));
    k_mc_bits<<<gb, 256, 0, s>>>(grid_.data(), static_cast<u32>(nseg), res[2], ntx, iso,
                                 bits_.data());
    WSIM_LAUNCH_CHECK();
    const McGrid M{res[0], res[1], res[2], ntx, static_cast<u32>(nseg), bits_.data()};
    k_mc_count<<<nb, kMeshThreads, 0, s>>>(M, dT, local_.data(), sums_.data());
    WSIM_LAUNCH_CHECK();
    k_mc_sums<<<1, kSumThreads, 0, s>>>(sums_.data(), nb, base, totals_.data());
    WSIM_LAUNCH_CHECK();
    u64 totals[2];
    read_back(totals, totals_.data(), sizeof(totals));
    const u64 nvert = totals[0], ntri = totals[1];
    if (nvert > 0xFFFFFFFFull || ntri > 0xFFFFFFFFull)
        fail(kOutOfRange, "SurfaceMesher: more than 2^32 - 1 elements");
    fit(verts_, 3 * std::max<u64>(nvert, 1));
    fit(tris_, 3 * std::max<u64>(ntri, 1));
    const bool post = P.smooth_post_iters > 0 && nvert > 0;
    if (post) {
        if (nv > (1ull << 30)) fail(kOutOfRange, "SurfaceMesher: grid too large for smoothing");
        fit(vpt_, nvert);
        for (auto& b : vd_) fit(b, 3 * nvert);
    }
    if (nvert) {
        k_mc_vertices<<<nb, kMeshThreads, 0, s>>>(
            grid_.data(), G, M, iso, local_.data(), sums_.data(), base, emask_.data(), eoff_.data(),
            verts_.data(), post ? vd_[0].data() : nullptr, post ? vpt_.data() : nullptr);
        WSIM_LAUNCH_CHECK();
        k_mc_triangles<<<nb, kMeshThreads, 0, s>>>(M, dT, local_.data(), sums_.data(), base,
                                                   emask_.data(), eoff_.data(), tris_.data());
        WSIM_LAUNCH_CHECK();
    }
    // 7. Laplacian mesh smoothing (:138-139)
    if (post) {
        fit(adj_, nvert * kAdjCap);
        fit(deg_, nvert);
        fit(adj_over_, kPartLine + kPartCounts);  // the overflow flag, counts of the list
        WSIM_HIP(hipMemsetAsync(adj_over_.data(), 0, (kPartLine + kPartCounts) * sizeof(u32), s));
        const u32 ga = static_cast<u32>((nvert + 255) / 256);
        // listed vertices lie in the smoothing's second buffer until its first pass:
        // 24 bytes a vertex, and from kAdjSplit on all parts are full but one round
        static_assert(kAdjSplit >= kParts * 256, "parts of whole workgroups fit in the buffer");
        const SplitList more{adj_over_.data() + kPartLine, reinterpret_cast<u32*>(vd_[1].data()),
                             part_capacity(ga, 256)};
        auto neighbours = [&](auto mode, u32 blocks) {
            k_mc_adjacency<decltype(mode)::value><<<blocks, 256, 0, s>>>(
                M, dT, nvert, vpt_.data(), emask_.data(), eoff_.data(), adj_.data(), deg_.data(),
                more, adj_over_.data());
            WSIM_LAUNCH_CHECK();
        };
        if (nvert < kAdjSplit) {
            neighbours(std::integral_constant<int, kAdjAll>{}, ga);
        } else {
            neighbours(std::integral_constant<int, kAdjFirst>{}, ga);
            neighbours(std::integral_constant<int, kAdjRest>{}, 2048);
        }
        const u64 n3 = 3 * nvert;
        const u32 g3 = static_cast<u32>((n3 + kMeshThreads - 1) / kMeshThreads);
        const u32 g1 = static_cast<u32>((nvert + kMeshThreads - 1) / kMeshThreads);
        int cur = 0;
        for (int it = 0; it < P.smooth_post_iters; ++it) {
            k_mesh_laplacian<<<g1, kMeshThreads, 0, s>>>(vd_[cur].data(), nvert, adj_.data(),
                                                         deg_.data(), vd_[cur ^ 1].data());
            WSIM_LAUNCH_CHECK();
            cur ^= 1;
        }
        k_verts_narrow<<<g3, kMeshThreads, 0, s>>>(vd_[cur].data(), n3, verts_.data());
        WSIM_LAUNCH_CHECK();
        u32 over = 0;  // (the lists are cut at their capacity, so the passes above stay in bounds)
        read_back(&over, adj_over_.data(), sizeof(u32));
        if (over) fail(kRuntimeError, "SurfaceMesher: a vertex with more than 24 neighbours");
    }
    WSIM_HIP(hipStreamSynchronize(s));
    info_.n_vertices = nvert;
    info_.n_triangles = ntri;
}

}  // namespace wsim
