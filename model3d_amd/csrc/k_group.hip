// k_group.hip -- GroupTriangles (GroupBounders, model3d/bvh.go:118-156,
// 219-292) on the device: the triangle order that SaveGroupedSTL writes
// (mesh.go:721-743) and that GroupedTrianglesToCollider expects.
//
// The reference sorts the triangles three times by their boxes' midpoints
// (one order per axis), then recursively cuts each node's range at n / 2
// along the axis whose two halves' box areas sum least, stably partitioning
// the other two orders by the halves; a node of one or two triangles is
// left in x order.  Here the recursion runs level by level over all nodes
// at once: the node of position p at level L is found by halving [0, n) L
// times, so no node table is kept.  Per level: the axis of every node (box
// reductions over its two halves in each order), a flag per triangle (in
// the first half along its node's axis), and a stable partition of each
// order inside its nodes (ranks of the flags).  Once a node's triangles fit a
// block's LDS, one block takes it through all its remaining levels there.
//
// A level of a few hundred thousand triangles is bound by its launches, not
// by its traffic: with a gather, a library scan and a scatter per order, 18
// levels of 203k triangles took 1.37 ms in 300 launches.  Here the LEVELS
// levels above GROUP_LOCAL triangles a node (8) take two launches for the
// three partitions (the flagged triangles before a node follow from the sizes
// alone), and the rest one kernel: 0.70 ms in 49 launches.  The initial sort
// is a stable radix sort of the three axes' keys at once, so equal midpoints
// stay in index order (the reference's sort.Slice leaves their order
// unspecified).
#include <hipcub/hipcub.hpp>

#include "launch.h"
#include "rect_collide.h"

namespace mc3d {
namespace {

// A double as a key whose unsigned order is the numeric order (-0 as +0,
// NaN last).
__device__ __forceinline__ uint64_t order_key(double x) {
    if (isnan(x)) return ~0ull;
    if (x == 0) x = 0;
    const uint64_t u = (uint64_t)__double_as_longlong(x);
    return (u >> 63) ? ~u : (u | (1ull << 63));
}
__device__ __forceinline__ double key_double(uint64_t k) {
    return __longlong_as_double((long long)((k >> 63) ? (k & ~(1ull << 63)) : ~k));
}

// The node of position p at level L: [lo, hi) after L halvings of [0, n)
// (the first half is the n / 2 smallest positions).
__device__ __forceinline__ uint32_t node_of(uint32_t p, uint32_t n, int L, uint32_t &lo, uint32_t &hi) {
    lo = 0, hi = n;
    uint32_t k = 0;
    for (int l = 0; l < L; l++) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (p < mid) hi = mid, k = 2 * k;
        else lo = mid, k = 2 * k + 1;
    }
    return k;
}
// The range of node k at level L.
__device__ __forceinline__ void node_range(uint32_t k, uint32_t n, int L, uint32_t &lo, uint32_t &hi) {
    lo = 0, hi = n;
    for (int l = L - 1; l >= 0; l--) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if ((k >> l) & 1u) lo = mid;
        else hi = mid;
    }
}

// Triangle boxes (Triangle.Min / Max, primitives.go:35-43), and each axis's
// midpoint keys with their triangles (axis * step + triangle).
__global__ __launch_bounds__(256) void k_grp_boxes(const double *__restrict__ verts, const uint32_t *__restrict__ tris,
                                                   uint32_t n, GroupBox *__restrict__ box, uint64_t *__restrict__ keys,
                                                   uint32_t *__restrict__ vals, uint32_t step) {
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        const double *p[3];
        for (int k = 0; k < 3; k++) p[k] = verts + 3 * (tris ? (size_t)tris[3 * (size_t)t + k] : 3 * (size_t)t + k);
        GroupBox b;
        for (int a = 0; a < 3; a++) {
            b.mn[a] = rc::go_min(rc::go_min(p[0][a], p[1][a]), p[2][a]);
            b.mx[a] = rc::go_max(rc::go_max(p[0][a], p[1][a]), p[2][a]);
            keys[(size_t)a * n + t] = order_key((b.mn[a] + b.mx[a]) * 0.5);  // Coord3D.Mid, coords.go:196-198
            vals[(size_t)a * n + t] = (uint32_t)a * step + t;
        }
        box[t] = b;
    }
}

// boundsArea (bvh.go:289-292) of a box
__device__ __forceinline__ double bounds_area(const double *mn, const double *mx) {
    const double dx = mx[0] + -mn[0], dy = mx[1] + -mn[1], dz = mx[2] + -mn[2];
    return 2 * (dx * (dy + dz) + dy * dz);
}

// multipleBoundsArea (bvh.go:257-287) starts from its first box and takes
// over what compares less or greater: a NaN of the first box stays, and any
// other is passed over.
__device__ __forceinline__ void keep_nan(const double *first_mn, const double *first_mx, double *mn, double *mx) {
    for (int c = 0; c < 3; c++) {
        if (isnan(first_mn[c])) mn[c] = first_mn[c];
        if (isnan(first_mx[c])) mx[c] = first_mx[c];
    }
}

// The node's axis (bestSplitAxis, bvh.go:219-236) from its halves' areas,
// area[2 * axis + half].
__device__ __forceinline__ uint8_t best_axis(const double *area) {
    int axis = 0;
    double best = area[0] + area[1];
    for (int a = 1; a < 3; a++) {
        const double v = area[2 * a] + area[2 * a + 1];
        if (v < best) best = v, axis = a;
    }
    return (uint8_t)axis;
}

// Every position of the three orders folds its box into its node half's slot
// (36 ordered keys per node: axis, half, min xyz, max xyz) with atomic min /
// max.  A block takes GRP_RUN * 256 consecutive positions of an order, 256 at
// a time: waves whose positions all lie in one node half fold them first, and
// while that half stays the block's they are kept and go out once a block (a
// few hundred atomics on one slot are what the top levels would wait for).
// The min and max leave NaN out, so they do not depend on the order (only the
// sign of a zero might, and it cannot change an area comparison).
constexpr int GRP_RUN = 8;

__device__ __forceinline__ void flush_box(unsigned long long *slot, const double *mn, const double *mx) {
    for (int c = 0; c < 3; c++) {
        atomicMin(&slot[c], (unsigned long long)order_key(mn[c]));
        atomicMax(&slot[3 + c], (unsigned long long)order_key(mx[c]));
    }
}

__global__ __launch_bounds__(256) void k_grp_fold(GroupLevel G, unsigned long long *__restrict__ slots) {
    __shared__ double part[4][6];
    __shared__ uint32_t part_key[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, a = (int)blockIdx.y;
    const uint32_t chunk = GRP_RUN * 256, nchunks = (G.n + chunk - 1) / chunk;
    auto slot = [&](uint32_t key) { return slots + (size_t)(key >> 1) * 36 + a * 12 + (key & 1) * 6; };
    for (uint32_t b = blockIdx.x; b < nchunks; b += gridDim.x) {
        uint32_t cur = ~0u;  // the wave's node half so far, its boxes folded a lane each
        double mn[3], mx[3];
        auto reduce = [&]() {
            for (int d = 32; d >= 1; d >>= 1)
                for (int c = 0; c < 3; c++) {
                    mn[c] = fmin(mn[c], __shfl_xor(mn[c], d, 64));
                    mx[c] = fmax(mx[c], __shfl_xor(mx[c], d, 64));
                }
        };
        uint32_t tri[GRP_RUN];
        for (int i = 0; i < GRP_RUN; i++) {
            const uint32_t p = b * chunk + (uint32_t)i * 256 + threadIdx.x;
            tri[i] = p < G.n ? G.perm[a][p] : ~0u;
        }
        for (int i = 0; i < GRP_RUN; i++) {
            const uint32_t p = b * chunk + (uint32_t)i * 256 + threadIdx.x;
            const bool have = tri[i] != ~0u;
            if (!__ballot(have)) break;
            const GroupBox box = G.box[have ? tri[i] : 0];
            uint32_t lo, hi, key = ~0u;
            if (have) {
                const uint32_t k = node_of(p, G.n, G.L, lo, hi);
                key = 2 * k + (p >= lo + (hi - lo) / 2);
            }
            const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)key);  // (lane 0 has one if any has)
            if (__ballot(have && key != first)) {  // several halves: straight to their slots
                if (cur != ~0u) {
                    reduce();
                    if (lane == 0) flush_box(slot(cur), mn, mx);
                    cur = ~0u;
                }
                if (have) {
                    for (int c = 0; c < 3; c++) mn[c] = fmin(INFINITY, box.mn[c]), mx[c] = fmax(-INFINITY, box.mx[c]);
                    flush_box(slot(key), mn, mx);
                }
                continue;
            }
            if (first != cur) {
                if (cur != ~0u) {
                    reduce();
                    if (lane == 0) flush_box(slot(cur), mn, mx);
                }
                cur = first;
                for (int c = 0; c < 3; c++) mn[c] = INFINITY, mx[c] = -INFINITY;
            }
            if (have)
                for (int c = 0; c < 3; c++) mn[c] = fmin(mn[c], box.mn[c]), mx[c] = fmax(mx[c], box.mx[c]);
        }
        // the waves' last halves, as one where they are the same
        if (cur != ~0u) reduce();
        __syncthreads();
        if (lane == 0) {
            part_key[wave] = cur;
            for (int c = 0; c < 3; c++) part[wave][c] = mn[c], part[wave][3 + c] = mx[c];
        }
        __syncthreads();
        if (lane == 0 && cur != ~0u) {
            bool mine = true;  // the first wave with this half takes the others'
            for (int w = 0; w < wave; w++) mine = mine && part_key[w] != cur;
            if (mine) {
                for (int w = wave + 1; w < 4; w++)
                    if (part_key[w] == cur)
                        for (int c = 0; c < 3; c++) mn[c] = fmin(mn[c], part[w][c]), mx[c] = fmax(mx[c], part[w][3 + c]);
                flush_box(slot(cur), mn, mx);
            }
        }
    }
}

__global__ __launch_bounds__(256) void k_grp_slots_init(unsigned long long *__restrict__ slots, uint32_t nodes) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nodes * 36; i += gridDim.x * blockDim.x)
        slots[i] = (i % 6) < 3 ? ~0ull : 0ull;
}

__global__ __launch_bounds__(256) void k_grp_axis_slots(GroupLevel G, const unsigned long long *__restrict__ slots) {
    const uint32_t nodes = 1u << G.L;
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < nodes; k += gridDim.x * blockDim.x) {
        uint32_t lo, hi;
        node_range(k, G.n, G.L, lo, hi);
        if (hi - lo <= 2) {
            G.axis[k] = 0;
            continue;
        }
        const unsigned long long *s = slots + (size_t)k * 36;
        double area[6];
        for (int q = 0; q < 6; q++) {
            double mn[3], mx[3];
            for (int c = 0; c < 3; c++) mn[c] = key_double(s[q * 6 + c]), mx[c] = key_double(s[q * 6 + 3 + c]);
            const GroupBox &first = G.box[G.perm[q / 2][q & 1 ? lo + (hi - lo) / 2 : lo]];
            keep_nan(first.mn, first.mx, mn, mx);
            area[q] = bounds_area(mn, mx);
        }
        G.axis[k] = best_axis(area);
    }
}

// flag[t] = 1 for the triangles in the first half of their node along the
// node's axis (splitBounders, bvh.go:159-217).
__global__ __launch_bounds__(256) void k_grp_flags(GroupLevel G) {
    each_order_entry(G.n, blockIdx.x * (uint64_t)blockDim.x + threadIdx.x, (uint64_t)gridDim.x * blockDim.x, [&](int a, uint32_t p) {
        uint32_t lo, hi;
        const uint32_t k = node_of(p, G.n, G.L, lo, hi);
        if (G.axis[k] == a) G.flag[G.perm[a][p]] = p < lo + (hi - lo) / 2;
    });
}

// Triangles flagged in the nodes of level L that lie before position lo, the
// start of one of them: a subtree of s triangles, d levels above its nodes,
// has (s mod 2^d) nodes of one more than s / 2^d, and a node of m flags m / 2.
__device__ __forceinline__ uint32_t flagged_in(uint32_t s, int d) {
    const uint32_t q = s >> d, r = s & ((1u << d) - 1);
    return ((1u << d) - r) * (q / 2) + r * ((q + 1) / 2);
}
// node_of, and the flags before the node.
__device__ __forceinline__ void node_flags(uint32_t p, uint32_t n, int L, uint32_t &lo, uint32_t &hi, uint32_t &before) {
    lo = 0, hi = n, before = 0;
    for (int l = 0; l < L; l++) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if (p < mid) hi = mid;
        else before += flagged_in(mid - lo, L - 1 - l), lo = mid;
    }
}

// Positions of a partition tile: GRP_ITEMS consecutive ones a thread.
constexpr int GRP_ITEMS = 4, GRP_TILE = 256 * GRP_ITEMS;
// Up to this many tiles an order, a tile adds up the counts before it itself
// (more are scanned first).
constexpr uint32_t GRP_SUM_TILES = 2048;

__device__ __forceinline__ uint32_t wave_inclusive(uint32_t v) {
    const int lane = threadIdx.x & 63;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

// Flagged triangles of every tile of the three orders.
__global__ __launch_bounds__(256) void k_grp_count(GroupLevel G, uint32_t ntiles, uint32_t *__restrict__ counts) {
    __shared__ uint32_t sh[4];
    const int a = (int)blockIdx.y;
    for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        uint32_t c = 0;
        for (int i = 0; i < GRP_ITEMS; i++) {
            const uint32_t p = t * GRP_TILE + (uint32_t)i * 256 + threadIdx.x;
            const bool f = p < G.n && G.flag[G.perm[a][p]];
            c += (uint32_t)__popcll(__ballot(f));
        }
        __syncthreads();
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = c;
        __syncthreads();
        if (threadIdx.x == 0) counts[(size_t)a * ntiles + t] = sh[0] + sh[1] + sh[2] + sh[3];
    }
}

// Exclusive scan of each order's tile counts in place (a block an order).
__global__ __launch_bounds__(1024) void k_grp_scan_tiles(uint32_t ntiles, uint32_t *__restrict__ counts) {
    __shared__ uint32_t sh[16];
    uint32_t *c = counts + (size_t)blockIdx.x * ntiles;
    uint32_t carry = 0;
    for (uint32_t t0 = 0; t0 < ntiles; t0 += 1024) {
        const uint32_t t = t0 + threadIdx.x, v = t < ntiles ? c[t] : 0u;
        const uint32_t inc = wave_inclusive(v);
        __syncthreads();
        if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6] = inc;
        __syncthreads();
        uint32_t pre = carry, all = 0;
        for (int w = 0; w < 16; w++) pre += w < (int)(threadIdx.x >> 6) ? sh[w] : 0u, all += sh[w];
        if (t < ntiles) c[t] = pre + inc - v;
        carry += all;
    }
}

// Entries of the tiles before tile t of a row of counts (every thread's).
__device__ __forceinline__ uint32_t tile_base(const uint32_t *c, uint32_t t, bool scanned, uint32_t *sh) {
    if (scanned) return c[t];
    uint32_t base = 0;
    for (uint32_t i = threadIdx.x; i < t; i += 256) base += c[i];
    for (int d = 32; d; d >>= 1) base += __shfl_xor(base, d, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = base;
    __syncthreads();
    return sh[0] + sh[1] + sh[2] + sh[3];
}

// The three orders out of one sort of all 3 n keys (values axis * n +
// triangle): entries of every axis in a tile, then each to its place.
__device__ __forceinline__ int axis_of(uint32_t v, uint32_t n) { return v >= n ? (v >= 2 * n ? 2 : 1) : 0; }

__global__ __launch_bounds__(256) void k_grp_split_count(const uint32_t *__restrict__ vals, uint32_t n, uint32_t ntiles,
                                                         uint32_t *__restrict__ counts) {
    __shared__ uint32_t sh[3][4];
    const int wave = threadIdx.x >> 6;
    for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        uint32_t c[3] = {0, 0, 0};
        for (int i = 0; i < GRP_ITEMS; i++) {
            const uint32_t p = t * GRP_TILE + (uint32_t)i * 256 + threadIdx.x;
            const int a = p < 3 * n ? axis_of(vals[p], n) : 3;
            for (int q = 0; q < 3; q++) c[q] += (uint32_t)__popcll(__ballot(a == q));
        }
        __syncthreads();
        if ((threadIdx.x & 63) == 0)
            for (int q = 0; q < 3; q++) sh[q][wave] = c[q];
        __syncthreads();
        if (threadIdx.x < 3) {
            const uint32_t *s = sh[threadIdx.x];
            counts[(size_t)threadIdx.x * ntiles + t] = s[0] + s[1] + s[2] + s[3];
        }
    }
}

__global__ __launch_bounds__(256) void k_grp_split(const uint32_t *__restrict__ vals, uint32_t n, uint32_t ntiles,
                                                   const uint32_t *__restrict__ counts, bool scanned,
                                                   uint32_t *__restrict__ out) {
    __shared__ uint32_t sh[3][4], sh_base[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        uint32_t pos[3], v[GRP_ITEMS], sum[3] = {0, 0, 0}, inc[3];
        const uint32_t p0 = t * GRP_TILE + threadIdx.x * GRP_ITEMS;
        for (int i = 0; i < GRP_ITEMS; i++) v[i] = p0 + i < 3 * n ? vals[p0 + i] : ~0u;
        for (int i = 0; i < GRP_ITEMS; i++)
            for (int q = 0; q < 3; q++) sum[q] += v[i] != ~0u && axis_of(v[i], n) == q;
        // (a tile's entries lie before it in one order or another: the third
        // order's follow from the first two)
        pos[0] = tile_base(counts, t, scanned, sh_base);
        pos[1] = tile_base(counts + ntiles, t, scanned, sh_base);
        pos[2] = t * GRP_TILE - pos[0] - pos[1];
        for (int q = 0; q < 3; q++) inc[q] = wave_inclusive(sum[q]);
        if (lane == 63)
            for (int q = 0; q < 3; q++) sh[q][wave] = inc[q];
        __syncthreads();
        for (int q = 0; q < 3; q++) {
            for (int w = 0; w < wave; w++) pos[q] += sh[q][w];
            pos[q] += inc[q] - sum[q];
        }
        for (int i = 0; i < GRP_ITEMS; i++) {
            if (v[i] == ~0u) break;
            const int a = axis_of(v[i], n);
            const uint32_t at = a == 0 ? pos[0] : a == 1 ? pos[1] : pos[2];
            for (int q = 0; q < 3; q++) pos[q] += a == q;
            out[(size_t)a * n + at] = v[i] - (uint32_t)a * n;
        }
        __syncthreads();
    }
}

// The stable partition of the three orders inside each node: flagged
// triangles first, each side in its previous order.
struct GroupOut {
    uint32_t *perm[3];
};
__global__ __launch_bounds__(256) void k_grp_partition(GroupLevel G, uint32_t ntiles, const uint32_t *__restrict__ counts,
                                                       bool scanned, GroupOut out) {
    __shared__ uint32_t sh[4];
    const int a = (int)blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t *c = counts + (size_t)a * ntiles;
    for (uint32_t t = blockIdx.x; t < ntiles; t += gridDim.x) {
        uint32_t base = tile_base(c, t, scanned, sh);
        uint32_t tri[GRP_ITEMS], f[GRP_ITEMS], sum = 0;
        const uint32_t p0 = t * GRP_TILE + threadIdx.x * GRP_ITEMS;
        for (int i = 0; i < GRP_ITEMS; i++) tri[i] = p0 + i < G.n ? G.perm[a][p0 + i] : 0u;
        for (int i = 0; i < GRP_ITEMS; i++) f[i] = p0 + i < G.n ? (uint32_t)G.flag[tri[i]] : 0u, sum += f[i];
        const uint32_t inc = wave_inclusive(sum);
        __syncthreads();
        if (lane == 63) sh[wave] = inc;
        __syncthreads();
        for (int w = 0; w < wave; w++) base += sh[w];
        uint32_t s = base + inc - sum;  // flags before p0
        uint32_t lo = 0, hi = 0, before = 0;
        for (int i = 0; i < GRP_ITEMS; i++) {
            const uint32_t p = p0 + i;
            if (p >= G.n) break;
            if (p >= hi) node_flags(p, G.n, G.L, lo, hi, before);
            const uint32_t mid = lo + (hi - lo) / 2, r = s - before;
            out.perm[a][f[i] ? lo + r : mid + (p - lo - r)] = tri[i];
            s += f[i];
        }
    }
}

// The rest of the recursion of the nodes of level G.L, at most GRP_LOCAL
// triangles each, a block a node: boxes and orders (as indices into the
// node's x order) in LDS, every level there.  Only the x order is wanted.
// inv: scratch, an entry per triangle.
constexpr int GRP_THREADS = 1024, GRP_PER = GROUP_LOCAL / GRP_THREADS;
__global__ __launch_bounds__(GRP_THREADS) void k_grp_local(GroupLevel G, uint32_t *__restrict__ inv,
                                                           uint32_t *__restrict__ out) {
    __shared__ double bmn[3][GROUP_LOCAL], bmx[3][GROUP_LOCAL];
    __shared__ uint16_t ord_all[2][3][GROUP_LOCAL];
    __shared__ uint16_t rank[GROUP_LOCAL];
    __shared__ uint8_t flag[GROUP_LOCAL], axis[GROUP_LOCAL / 2];
    __shared__ double area[6 * 32];
    __shared__ uint32_t sh[GRP_THREADS / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (uint32_t k = blockIdx.x; k < (1u << G.L); k += gridDim.x) {
        uint32_t lo0, hi0;
        node_range(k, G.n, G.L, lo0, hi0);
        const int m = (int)(hi0 - lo0);
        __syncthreads();  // the previous node is done with the LDS
        for (int i = tid; i < m; i += GRP_THREADS) {
            const uint32_t t = G.perm[0][lo0 + i];
            const GroupBox b = G.box[t];
            for (int c = 0; c < 3; c++) bmn[c][i] = b.mn[c], bmx[c][i] = b.mx[c];
            ord_all[0][0][i] = (uint16_t)i;
            inv[t] = (uint32_t)i;
        }
        __threadfence_block();
        __syncthreads();
        for (int a = 1; a < 3; a++)
            for (int i = tid; i < m; i += GRP_THREADS)
                ord_all[0][a][i] = (uint16_t)__hip_atomic_load(&inv[G.perm[a][lo0 + i]], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __syncthreads();
        int cur = 0;
        for (int L = 0; ((m + (1 << L) - 1) >> L) > 2; L++) {
            uint16_t(*ord)[GROUP_LOCAL] = ord_all[cur], (*nxt)[GROUP_LOCAL] = ord_all[cur ^ 1];
            const uint32_t nodes = 1u << L;
            // 1. the nodes' axes
            if (nodes <= 32) {  // a wave per (node, axis, half)
                for (uint32_t q = (uint32_t)wave; q < 6 * nodes; q += GRP_THREADS / 64) {
                    uint32_t lo, hi;
                    node_range(q / 6, (uint32_t)m, L, lo, hi);
                    const uint32_t mid = lo + (hi - lo) / 2, a = (q % 6) / 2, s = q & 1 ? mid : lo, e = q & 1 ? hi : mid;
                    double mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
                    for (uint32_t p = s + lane; p < e; p += 64) {
                        const int i = ord[a][p];
                        for (int c = 0; c < 3; c++) mn[c] = fmin(mn[c], bmn[c][i]), mx[c] = fmax(mx[c], bmx[c][i]);
                    }
                    for (int d = 32; d; d >>= 1)
                        for (int c = 0; c < 3; c++) {
                            mn[c] = fmin(mn[c], __shfl_xor(mn[c], d, 64));
                            mx[c] = fmax(mx[c], __shfl_xor(mx[c], d, 64));
                        }
                    if (lane == 0) {
                        const int i = ord[a][s];
                        const double fmn[3] = {bmn[0][i], bmn[1][i], bmn[2][i]}, fmx[3] = {bmx[0][i], bmx[1][i], bmx[2][i]};
                        keep_nan(fmn, fmx, mn, mx);
                        area[q] = bounds_area(mn, mx);
                    }
                }
                __syncthreads();
                if ((uint32_t)tid < nodes) {
                    uint32_t lo, hi;
                    node_range(tid, (uint32_t)m, L, lo, hi);
                    axis[tid] = hi - lo <= 2 ? 0 : best_axis(area + 6 * tid);
                }
            } else {  // a thread per node
                for (uint32_t q = (uint32_t)tid; q < nodes; q += GRP_THREADS) {
                    uint32_t lo, hi;
                    node_range(q, (uint32_t)m, L, lo, hi);
                    double ar[6];
                    for (int h = 0; h < 6; h++) {
                        const uint32_t mid = lo + (hi - lo) / 2, s = h & 1 ? mid : lo, e = h & 1 ? hi : mid;
                        const int i0 = ord[h / 2][s];
                        double mn[3], mx[3];
                        for (int c = 0; c < 3; c++) mn[c] = bmn[c][i0], mx[c] = bmx[c][i0];
                        for (uint32_t p = s + 1; p < e; p++) {
                            const int i = ord[h / 2][p];
                            for (int c = 0; c < 3; c++) {
                                if (bmn[c][i] < mn[c]) mn[c] = bmn[c][i];
                                if (bmx[c][i] > mx[c]) mx[c] = bmx[c][i];
                            }
                        }
                        ar[h] = bounds_area(mn, mx);
                    }
                    axis[q] = hi - lo <= 2 ? 0 : best_axis(ar);
                }
            }
            __syncthreads();
            // 2. the flags, from each node's own axis
            for (int p = tid; p < m; p += GRP_THREADS) {
                uint32_t lo, hi;
                const uint32_t nd = node_of((uint32_t)p, (uint32_t)m, L, lo, hi);
                flag[ord[axis[nd]][p]] = (uint32_t)p < lo + (hi - lo) / 2;
            }
            __syncthreads();
            // 3. the partitions
            for (int a = 0; a < 3; a++) {
                uint32_t f[GRP_PER], sum = 0;
                for (int i = 0; i < GRP_PER; i++) {
                    const int p = tid * GRP_PER + i;
                    f[i] = p < m ? flag[ord[a][p]] : 0u;
                    sum += f[i];
                }
                const uint32_t inc = wave_inclusive(sum);
                if (lane == 63) sh[wave] = inc;
                __syncthreads();
                uint32_t s = inc - sum;
                for (int w = 0; w < wave; w++) s += sh[w];
                for (int i = 0; i < GRP_PER; i++) {
                    const int p = tid * GRP_PER + i;
                    if (p < m) rank[p] = (uint16_t)s;
                    s += f[i];
                }
                __syncthreads();
                for (int i = 0; i < GRP_PER; i++) {
                    const int p = tid * GRP_PER + i;
                    if (p >= m) break;
                    uint32_t lo, hi;
                    node_of((uint32_t)p, (uint32_t)m, L, lo, hi);
                    const uint32_t mid = lo + (hi - lo) / 2, r = (uint32_t)rank[p] - rank[lo];
                    nxt[a][f[i] ? lo + r : mid + ((uint32_t)p - lo - r)] = ord[a][p];
                }
                __syncthreads();
            }
            cur ^= 1;
        }
        // the node's triangles in their x order
        for (int i = tid; i < m; i += GRP_THREADS) out[lo0 + i] = G.perm[0][lo0 + ord_all[cur][0][i]];
    }
}

__global__ __launch_bounds__(256) void k_grp_apply(const uint32_t *__restrict__ tris, const uint32_t *__restrict__ perm,
                                                   uint32_t n, uint32_t *__restrict__ out) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < 3ull * n; i += (uint64_t)gridDim.x * blockDim.x)
        out[i] = tris[3 * (size_t)perm[i / 3] + i % 3];
}

}  // namespace

hipError_t launch_grp_apply(const uint32_t *tris, const uint32_t *perm, uint32_t n, uint32_t *out, hipStream_t st) {
    k_grp_apply<<<grid_for(3ull * n, 256, 8192), 256, 0, st>>>(tris, perm, n, out);
    return hipGetLastError();
}

hipError_t launch_grp_boxes(const double *verts, const uint32_t *tris, uint32_t n, GroupBox *box, uint64_t *keys,
                            uint32_t *vals, uint32_t step, hipStream_t st) {
    k_grp_boxes<<<grid_for(n, 256, 4096), 256, 0, st>>>(verts, tris, n, box, keys, vals, step);
    return hipGetLastError();
}

hipError_t launch_grp_split(const uint32_t *vals, uint32_t n, uint32_t *counts, uint32_t *out, hipStream_t st) {
    const uint32_t ntiles = grp_tiles(3 * n), blocks = std::min(ntiles, 8192u);
    const bool scanned = ntiles > GRP_SUM_TILES;
    k_grp_split_count<<<blocks, 256, 0, st>>>(vals, n, ntiles, counts);
    if (scanned) k_grp_scan_tiles<<<3, 1024, 0, st>>>(ntiles, counts);
    k_grp_split<<<blocks, 256, 0, st>>>(vals, n, ntiles, counts, scanned, out);
    return hipGetLastError();
}

hipError_t grp_sort(void *tmp, size_t &bytes, const uint64_t *keys_in, uint64_t *keys_out, const uint32_t *vals_in,
                    uint32_t *vals_out, uint32_t n, hipStream_t st) {
    return hipcub::DeviceRadixSort::SortPairs(tmp, bytes, keys_in, keys_out, vals_in, vals_out, (int)n, 0, 64, st);
}

hipError_t launch_grp_axis(const GroupLevel &G, unsigned long long *slots, hipStream_t st) {
    const uint32_t nodes = 1u << G.L;
    k_grp_slots_init<<<grid_for((uint64_t)nodes * 36, 256, 4096), 256, 0, st>>>(slots, nodes);
    const uint32_t chunks = (G.n + GRP_RUN * 256 - 1) / (GRP_RUN * 256);
    k_grp_fold<<<dim3(std::min(chunks, 8192u), 3), 256, 0, st>>>(G, slots);
    k_grp_axis_slots<<<grid_for(nodes, 256, 4096), 256, 0, st>>>(G, slots);
    return hipGetLastError();
}

hipError_t launch_grp_flags(const GroupLevel &G, hipStream_t st) {
    k_grp_flags<<<grid_for(3ull * G.n, 256, 8192), 256, 0, st>>>(G);
    return hipGetLastError();
}

uint32_t grp_tiles(uint32_t n) { return (n + GRP_TILE - 1) / GRP_TILE; }

hipError_t launch_grp_partition(const GroupLevel &G, uint32_t *counts, uint32_t *const out[3], hipStream_t st) {
    const uint32_t ntiles = grp_tiles(G.n);
    const dim3 grid(std::min(ntiles, 8192u), 3);
    const bool scanned = ntiles > GRP_SUM_TILES;
    k_grp_count<<<grid, 256, 0, st>>>(G, ntiles, counts);
    if (scanned) k_grp_scan_tiles<<<3, 1024, 0, st>>>(ntiles, counts);
    k_grp_partition<<<grid, 256, 0, st>>>(G, ntiles, counts, scanned, GroupOut{{out[0], out[1], out[2]}});
    return hipGetLastError();
}

hipError_t launch_grp_local(const GroupLevel &G, uint32_t *inv, uint32_t *out, hipStream_t st) {
    k_grp_local<<<std::min(1u << G.L, 65536u), GRP_THREADS, 0, st>>>(G, inv, out);
    return hipGetLastError();
}

}  // namespace mc3d
