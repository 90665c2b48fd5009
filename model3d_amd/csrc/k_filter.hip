// k_filter.hip -- MarchingCubesFilter's block recursion with a mesh
// collider's RectCollision as the filter (MarchingCubesC2F, and
// MarchingCubesSearchFilter with the library's rect collider), on the
// device.
//
//   MarchingCubesFilter / C2F                  model3d/mc.go:83-180
//   mcBlock (Bounds, Volume, Pieces, Split)    model3d/mc.go:724-797
//   MeshToCollider(...).RectCollision          model3d/collisions.go:138-142, 169-179, 344-356
//
// The collider's triangles are binned in a uniform 3D grid by their boxes;
// a rect's answer is the OR over the triangles of the cells it overlaps of
// "the triangle's box overlaps the rect and Triangle.RectCollision" -- the
// answer the collider's tree gives, whose every node box contains the boxes
// of the triangles below it.
//
// A leaf of the recursion (volume / 2 below 64) is accepted when it and
// every block above it are.  The splits do not depend on the filter, so a
// leaf is a path of halvings from the root, and all leaves are asked at once,
// a lane each: most are decided by summed-volume tables (no triangle listed
// in the rect's cells: rejected; a segment origin in a cell inside it:
// accepted, and with it every block above, whose rects contain the leaf's).
// Those left open are asked with Triangle.RectCollision, a wave each, and where
// the leaf is hit without an origin in it the blocks above it too: first of the
// triangle that hits the leaf, a lane a block.  The reference's two-stage
// recursion (first down to max(volume / 4096, 64), then each queued block down
// to 64) asks the same deterministic filter of the same blocks, so its accepted
// leaves are these.
//
// Level by level (a kernel per level, each waiting for the one above, four
// blocks a wave so that open ones did not wait for each other) a grid of
// 402^3 corners with 51k triangles took 1,660 us; here the leaves take 54 us
// (the mask's atomics) and the open ones 247 us, bound by the chain of
// loads to each batch of 64 listed triangles (list, box, triangle) at 2 waves
// per SIMD (240 registers, of the triangle test).  Cells of one coarse spacing
// instead of two list fewer triangles per rect (open 610 -> 460 us); the boxes
// kept from the binning reject most of a batch with six comparisons (460 -> 372
// us); the blocks above asked of one triangle, not each in turn of the mesh, 376
// -> 247 us.  A triangle as large as the grid leaves most leaves open: a list of a
// quarter of them, the rest asked by the waves that found them, took 5,400 us for
// twelve triangles on 202^3 corners (the levels 1,200 us; now 600).
#include "launch.h"
#include "rect_collide.h"

namespace mc3d {
namespace {

__device__ __forceinline__ void cell_range(double lo, double hi, double o, double inv, int n, int &c0, int &c1) {
    // clamped to the grid (a NaN bound: cell 0; such a rect overlaps no box)
    const double a = floor((lo - o) * inv), b = floor((hi - o) * inv);
    c0 = a >= 0 ? (a <= n - 1 ? (int)a : n - 1) : 0;
    c1 = b >= 0 ? (b <= n - 1 ? (int)b : n - 1) : 0;
}

// The cells of a triangle's box; false for a box with NaN bounds (such a
// triangle's box overlaps no rect).
__device__ __forceinline__ bool tri_cells(const RectGridDev &R, const GroupBox &b, int *c0, int *c1) {
    for (int a = 0; a < 3; a++) {
        if (isnan(b.mn[a]) || isnan(b.mx[a])) return false;
        cell_range(b.mn[a], b.mx[a], R.o[a], R.inv, R.n[a], c0[a], c1[a]);
    }
    return true;
}

__global__ __launch_bounds__(256) void k_rgrid_gather(const double *__restrict__ verts,
                                                      const uint32_t *__restrict__ tris, uint64_t nt,
                                                      double *__restrict__ out) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < 9 * nt;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t t = i / 9, r = i - 9 * t;
        out[i] = verts[3 * (uint64_t)tris[3 * t + r / 3] + r % 3];
    }
}

__global__ __launch_bounds__(256) void k_rgrid_count(RectGridDev R, GroupBox *__restrict__ box,
                                                     uint32_t *__restrict__ counts) {
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < R.ntris; t += gridDim.x * blockDim.x) {
        int c0[3], c1[3];
        GroupBox b;
        rc::tri_box(R.tris + 9 * (size_t)t, b.mn, b.mx);
        box[t] = b;
        if (!tri_cells(R, b, c0, c1)) continue;
        for (int z = c0[2]; z <= c1[2]; z++)
            for (int y = c0[1]; y <= c1[1]; y++)
                for (int x = c0[0]; x <= c1[0]; x++) atomicAdd(&counts[((size_t)z * R.n[1] + y) * R.n[0] + x], 1u);
    }
}

__global__ __launch_bounds__(256) void k_rgrid_fill(RectGridDev R, uint32_t *__restrict__ cursor,
                                                    uint32_t *__restrict__ cell_tris) {
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < R.ntris; t += gridDim.x * blockDim.x) {
        int c0[3], c1[3];
        if (!tri_cells(R, R.box[t], c0, c1)) continue;
        for (int z = c0[2]; z <= c1[2]; z++)
            for (int y = c0[1]; y <= c1[1]; y++)
                for (int x = c0[0]; x <= c1[0]; x++)
                    cell_tris[atomicAdd(&cursor[((size_t)z * R.n[1] + y) * R.n[0] + x], 1u)] = t;
    }
}

// Counts each segment origin (rc::origin_vertices) in its cell of the
// vertex grid; one outside the grid is not counted.
__global__ __launch_bounds__(256) void k_vgrid_count(RectGridDev R, uint32_t *__restrict__ vsat) {
    for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < R.ntris; t += gridDim.x * blockDim.x) {
        const double *p = R.tris + 9 * (size_t)t;
        bool origin[3];
        if (!rc::origin_vertices(p, origin)) continue;
        for (int k = 0; k < 3; k++) {
            if (!origin[k]) continue;
            int c[3];
            bool in = true;
            for (int a = 0; a < 3; a++) {
                const double f = floor((p[3 * k + a] - R.vo[a]) * R.vinv);
                in = in && f >= 0 && f < R.vn[a];
                c[a] = in ? (int)f : 0;
            }
            if (in) atomicAdd(&vsat[((size_t)c[2] * R.vn[1] + c[1]) * R.vn[0] + c[0]], 1u);
        }
    }
}

// Inclusive prefix sums along x (a wave per row), then y and z (a thread
// per column): the summed-volume table in place.
__global__ __launch_bounds__(256) void k_vsat_x(uint32_t *__restrict__ v, int n0, uint32_t rows) {
    const int lane = threadIdx.x & 63;
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, nw = (gridDim.x * blockDim.x) >> 6;
    for (uint32_t r = wave; r < rows; r += nw) {
        uint32_t *row = v + (size_t)r * n0, carry = 0;
        for (int x0 = 0; x0 < n0; x0 += 64) {
            const int x = x0 + lane;
            uint32_t s = x < n0 ? row[x] : 0u;
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t u = __shfl_up(s, d, 64);
                if (lane >= d) s += u;
            }
            if (x < n0) row[x] = s + carry;
            carry += __shfl(s, 63, 64);
        }
    }
}

__global__ __launch_bounds__(64) void k_vsat_yz(uint32_t *__restrict__ v, int n0, int n1, int n2, int axis) {
    // axis 1: columns (x, z) along y; axis 2: columns (x, y) along z
    const uint32_t ncol = (uint32_t)n0 * (axis == 1 ? n2 : n1);
    for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < ncol; c += gridDim.x * blockDim.x) {
        const uint32_t x = c % n0, w = c / n0;
        size_t i, step;
        int len;
        if (axis == 1) i = (size_t)w * n1 * n0 + x, step = n0, len = n1;
        else i = (size_t)w * n0 + x, step = (size_t)n0 * n1, len = n2;
        // eight loads in flight (a column is a chain of dependent additions,
        // and few columns run at once: one load at a time took 31 us for
        // 100^3 cells)
        uint32_t s = 0;
        int k = 0;
        for (; k + 8 <= len; k += 8, i += 8 * step) {
            uint32_t t[8];
            for (int j = 0; j < 8; j++) t[j] = v[i + j * step];
            for (int j = 0; j < 8; j++) v[i + j * step] = s += t[j];
        }
        for (; k < len; k++, i += step) v[i] = s += v[i];
    }
}

constexpr int RSCAN = 1024;  // cells per scan tile (one per thread of a 1024-thread block)

// Inclusive scan of one value per thread over a 1024-thread block.
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t *sh) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t u = __shfl_up(v, d, 64);
        if (lane >= d) v += u;
    }
    if (lane == 63) sh[wave] = v;
    __syncthreads();
    if (wave == 0) {
        uint32_t w = lane < 16 ? sh[lane] : 0;
        for (int d = 1; d < 16; d <<= 1) {
            const uint32_t u = __shfl_up(w, d, 64);
            if (lane >= d) w += u;
        }
        if (lane < 16) sh[lane] = w;
    }
    __syncthreads();
    return v + (wave ? sh[wave - 1] : 0);
}

// Tile sums of the counts.
__global__ __launch_bounds__(RSCAN) void k_rscan_tiles(const uint32_t *__restrict__ counts, uint32_t n,
                                                       uint32_t *__restrict__ tiles) {
    __shared__ uint32_t sh[16];
    const uint32_t i = blockIdx.x * RSCAN + threadIdx.x;
    const uint32_t s = block_scan(i < n ? counts[i] : 0u, sh);
    if (threadIdx.x == RSCAN - 1) tiles[blockIdx.x] = s;
}

// Exclusive scan of the tile sums (at most RSCAN tiles, one block).
__global__ __launch_bounds__(RSCAN) void k_rscan_top(uint32_t *__restrict__ tiles, uint32_t ntiles) {
    __shared__ uint32_t sh[16];
    const uint32_t v = threadIdx.x < ntiles ? tiles[threadIdx.x] : 0u;
    const uint32_t s = block_scan(v, sh);
    if (threadIdx.x < ntiles) tiles[threadIdx.x] = s - v;
}

// start[i] = cursor[i] = exclusive prefix of counts; start[n] = the total.
__global__ __launch_bounds__(RSCAN) void k_rscan_down(const uint32_t *__restrict__ counts, uint32_t n,
                                                      const uint32_t *__restrict__ tiles, uint32_t *__restrict__ start,
                                                      uint32_t *__restrict__ cursor) {
    __shared__ uint32_t sh[16];
    const uint32_t i = blockIdx.x * RSCAN + threadIdx.x;
    const uint32_t v = i < n ? counts[i] : 0u;
    const uint32_t s = block_scan(v, sh) + tiles[blockIdx.x];
    if (i < n) start[i] = cursor[i] = s - v;
    if (i == n - 1) start[n] = s;
}

// Candidate k of n in a scattered order (P prime and above n: a bijection),
// so that the first 64 lanes sample the whole rect, not its first rows.
__device__ __forceinline__ uint32_t scatter(uint32_t k, uint32_t n, uint64_t P) { return (uint32_t)(k * P % n); }

// Sum of the cells [lo, hi] from a summed-volume table of n[0] x n[1] x n[2].
__device__ __forceinline__ uint32_t table_sum(const uint32_t *__restrict__ t, const int *n, const int *lo, const int *hi) {
    auto S = [&](int x, int y, int z) -> uint32_t {
        if (x < 0 || y < 0 || z < 0) return 0u;
        return t[((size_t)z * n[1] + y) * n[0] + x];
    };
    const int x0 = lo[0] - 1, y0 = lo[1] - 1, z0 = lo[2] - 1, x1 = hi[0], y1 = hi[1], z1 = hi[2];
    return S(x1, y1, z1) - S(x0, y1, z1) - S(x1, y0, z1) - S(x1, y1, z0) + S(x0, y0, z1) + S(x0, y1, z0) + S(x1, y0, z0) -
           S(x0, y0, z0);
}

// A sure hit from the vertex table: a segment origin in a cell strictly
// inside the rect's cell range.  For such a vertex v in cell k on an axis,
// floor((v - o) * inv) = k > floor((mn - o) * inv) gives v > mn (the
// rounded subtraction and product are monotone), and k < floor((mx - o) *
// inv) gives v < mx; a vertex inside makes the collision (rc::vertex_inside).
__device__ __forceinline__ bool sure_hit(const RectGridDev &R, const double *mn, const double *mx) {
    if (!R.vsat) return false;
    int lo[3], hi[3];
    for (int a = 0; a < 3; a++) {
        if (isnan(mn[a]) || isnan(mx[a])) return false;
        int c0, c1;
        cell_range(mn[a], mx[a], R.vo[a], R.vinv, R.vn[a], c0, c1);
        lo[a] = c0 + 1, hi[a] = c1 - 1;  // (clamping only narrows the range)
        if (hi[a] < lo[a]) return false;
    }
    return table_sum(R.vsat, R.vn, lo, hi) != 0;
}

// No triangle is listed in the rect's cells: the rect overlaps no triangle's
// box (cell_range is monotone, so overlapping boxes share a cell).
__device__ __forceinline__ bool sure_miss(const RectGridDev &R, const double *mn, const double *mx) {
    int c0[3], c1[3];
    for (int a = 0; a < 3; a++) {
        cell_range(mn[a], mx[a], R.o[a], R.inv, R.n[a], c0[a], c1[a]);
        if (c1[a] < c0[a]) return true;  // min above max: the rect overlaps no box
    }
    return table_sum(R.csat, R.n, c0, c1) == 0;
}

// rc::box_overlap for boxes without NaN (none else is listed; a NaN on
// either side compares false, which is its answer too).
__device__ __forceinline__ bool boxes_overlap(const double *mn, const double *mx, const GroupBox &b) {
    return mn[0] <= b.mx[0] && b.mn[0] <= mx[0] && mn[1] <= b.mx[1] && b.mn[1] <= mx[1] && mn[2] <= b.mx[2] &&
           b.mn[2] <= mx[2] && mn[0] <= mx[0] && mn[1] <= mx[1] && mn[2] <= mx[2];
}

template <class T>
__device__ __forceinline__ T lane_value(T v, int j) {
    return __shfl(v, j, 64);
}

// One triangle's part of RectCollision for [mn, mx]: 0 no, 1 yes, 2 yes by a
// segment origin inside, which is inside every larger rect too.
__device__ __forceinline__ int tri_hits(const RectGridDev &R, uint32_t tri, const double *mn, const double *mx) {
    const double *p = R.tris + 9 * (size_t)tri;
    const rc::V v[3] = {rc::mk(p[0], p[1], p[2]), rc::mk(p[3], p[4], p[5]), rc::mk(p[6], p[7], p[8])};
    return rc::vertex_inside(p, mn, mx) ? 2 : (rc::tri_rect(v, mn, mx) ? 1 : 0);
}

// RectCollision of the mesh for [mn, mx] where the vertex table gave no sure
// hit, asked by a whole wave (the answer is wave-uniform, as tri_hits'; by: a
// triangle that hits): every candidate triangle tested once -- the triangles binned in the cells the rect
// overlaps, taken 64 at a time (each (y, z) row of those cells is one run
// of the cell lists; a triangle listed in several of the rect's cells is
// tested at the first of them), or, for a rect over more cells than half
// the triangles, all triangles in a scattered order.
__device__ int rect_hits(const RectGridDev &R, const double *mn, const double *mx, uint32_t &by) {
    const int lane = threadIdx.x & 63;
    int c0[3], c1[3];
    for (int a = 0; a < 3; a++) {
        cell_range(mn[a], mx[a], R.o[a], R.inv, R.n[a], c0[a], c1[a]);
        if (c1[a] < c0[a]) return 0;  // min above max: the rect overlaps no box
    }
    const uint32_t lx = c1[0] - c0[0] + 1, ly = c1[1] - c0[1] + 1, lz = c1[2] - c0[2] + 1;
    const uint64_t ncell = (uint64_t)lx * ly * lz;
    if (2 * ncell > R.ntris) {
        for (uint32_t t0 = 0; t0 < R.ntris; t0 += 64) {
            int h = 0;
            uint32_t t = 0;
            if (t0 + lane < R.ntris) {
                t = scatter(t0 + lane, R.ntris, 4294967291ull);
                if (boxes_overlap(mn, mx, R.box[t])) h = tri_hits(R, t, mn, mx);
            }
            if (const uint64_t m = __ballot(h != 0)) {
                by = lane_value(t, __ffsll((unsigned long long)m) - 1);
                return __ballot(h == 2) ? 2 : 1;
            }
        }
        return 0;
    }
    const uint32_t nrows = ly * lz;
    for (uint32_t r0 = 0; r0 < nrows; r0 += 64) {
        // lane i: row r0 + i, its run [a, a + len) of cell_tris
        const uint32_t r = r0 + lane;
        uint32_t a = 0, len = 0;
        int ry = 0, rz = 0;
        if (r < nrows) {
            ry = c0[1] + (int)(r % ly), rz = c0[2] + (int)(r / ly);
            const size_t row = ((size_t)rz * R.n[1] + ry) * R.n[0];
            a = R.cell_start[row + c0[0]];
            len = R.cell_start[row + c1[0] + 1] - a;
        }
        uint32_t incl = len;
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t u = __shfl_up(incl, d, 64);
            if (lane >= d) incl += u;
        }
        const uint32_t excl = incl - len, total = __shfl(incl, 63, 64);
        for (uint32_t e0 = 0; e0 < total; e0 += 64) {
            const uint32_t e = e0 + lane;
            // the row holding entry e: the first lane j with incl_j > e
            int lo = 0, hi = 63;
            for (int k = 0; k < 6; k++) {
                const int mid = (lo + hi) >> 1;
                if (__shfl(incl, mid, 64) > e) hi = mid;
                else lo = mid + 1;
            }
            const uint32_t aj = __shfl(a, lo, 64), xj = __shfl(excl, lo, 64);
            const int yj = __shfl(ry, lo, 64), zj = __shfl(rz, lo, 64);
            int h = 0;
            uint32_t tri = 0;
            if (e < total) {
                const uint32_t idx = aj + (e - xj);
                tri = R.cell_tris[idx];
                const GroupBox tb = R.box[tri];
                if (boxes_overlap(mn, mx, tb)) {
                    // the first of the rect's cells that list it: row (y, z)
                    // at max(its first cell, the rect's), then the cell's run
                    int t0[3], t1[3];
                    for (int ax = 0; ax < 3; ax++) cell_range(tb.mn[ax], tb.mx[ax], R.o[ax], R.inv, R.n[ax], t0[ax], t1[ax]);
                    if (yj == max(t0[1], c0[1]) && zj == max(t0[2], c0[2])) {
                        const size_t cf = ((size_t)zj * R.n[1] + yj) * R.n[0] + max(t0[0], c0[0]);
                        if (idx >= R.cell_start[cf] && idx < R.cell_start[cf + 1]) h = tri_hits(R, tri, mn, mx);
                    }
                }
            }
            if (const uint64_t m = __ballot(h != 0)) {
                by = lane_value(tri, __ffsll((unsigned long long)m) - 1);
                return __ballot(h == 2) ? 2 : 1;
            }
        }
    }
    return 0;
}

// mcBlock.Pieces(64, ...) stops at this block (mc.go:760-775).
__device__ __forceinline__ bool is_leaf(const FBlock &b) {
    return (int64_t)(b.mx[0] - b.mn[0]) * (b.mx[1] - b.mn[1]) * (b.mx[2] - b.mn[2]) / 2 < 64;
}

// mcBlock.Split (mc.go:777-797): a half of the longest axis (y, then z on
// ties with x).
__device__ __forceinline__ void halve(FBlock &b, bool second) {
    const int lx = b.mx[0] - b.mn[0], ly = b.mx[1] - b.mn[1], lz = b.mx[2] - b.mn[2];
    int axis = 0;
    if (ly >= lx && ly >= lz) axis = 1;
    else if (lz >= lx && lz >= ly) axis = 2;
    for (int a = 0; a < 3; a++)
        if (a == axis) {
            const int mid = (b.mx[a] + b.mn[a]) / 2;
            if (second) b.mn[a] = mid;
            else b.mx[a] = mid;
        }
}

// mcBlock.Bounds(epsilon) (mc.go:736-740), then the filter's
// Rect.Expand(extra) (shapes.go:339-344; extra 0: the rect itself).
__device__ __forceinline__ void block_rect(const BlockFilter &F, const FBlock &b, double *mn, double *mx) {
    const double *ax[3] = {F.xs, F.ys, F.zs};
    for (int a = 0; a < 3; a++) {
        mn[a] = (ax[a][b.mn[a]] + -F.eps) + -F.extra;
        mx[a] = (ax[a][b.mx[a]] + F.eps) + F.extra;
    }
}

// Cubes [x0, x1) of a row into the mask.
__device__ __forceinline__ void set_cubes(unsigned long long *row, int x0, int x1) {
    for (int x = x0; x < x1;) {
        const int w = x >> 6, lo = x & 63, hi = min(64, x1 - (w << 6));
        const uint64_t m = (hi >= 64 ? ~0ull : ((1ull << hi) - 1)) & (~0ull << lo);
        atomicOr(&row[w], (unsigned long long)m);
        x = (w << 6) + hi;
    }
}

__device__ __forceinline__ unsigned long long *keep_row(const BlockFilter &F, int y, int z) {
    return (unsigned long long *)F.keep + ((size_t)z * F.ny + y) * F.W;
}

// The leaf at the end of `path` (bit depth - 1 first; one path for the
// wave), asked by the whole wave.
__device__ void open_leaf(const BlockFilter &F, const FBlock &root, int depth, uint64_t path) {
    const int lane = threadIdx.x & 63;
    path = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)path) |
           ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(path >> 32)) << 32);
    FBlock b = root;
    int leaf = 0;  // its depth
    for (; leaf < depth && !is_leaf(b); leaf++) halve(b, (path >> (depth - 1 - leaf)) & 1);
    double mn[3], mx[3];
    block_rect(F, b, mn, mx);
    // The leaf, then (lane i: i halvings down) the blocks above it: almost always
    // the triangle that hits the leaf hits them all, each asked of it by its own
    // lane; one that it does not hit, and whose rect holds no other that certainly
    // is hit, is asked of the mesh.
    uint64_t ask = 0;
    double amn[3], amx[3];
    for (int at = leaf;;) {
        uint32_t by = 0;
        const int hit = rect_hits(F.R, mn, mx, by);
        if (!hit) return;
        if (hit == 2) break;
        if (at == leaf) {
            FBlock u = root;
            for (int d = 0; d < min(lane, leaf); d++) halve(u, (path >> (depth - 1 - d)) & 1);
            block_rect(F, u, amn, amx);
            const int h = sure_hit(F.R, amn, amx) ? 2 : (boxes_overlap(amn, amx, F.R.box[by]) ? tri_hits(F.R, by, amn, amx) : 0);
            ask = __ballot(lane < leaf && h == 0);
            const uint64_t sure = __ballot(lane < leaf && h == 2);
            if (sure) ask &= ~(~0ull >> __clzll((long long)sure));
        }
        if (!ask) break;
        at = 63 - __clzll((long long)ask);
        ask &= ~(1ull << at);
        for (int a = 0; a < 3; a++) mn[a] = lane_value(amn[a], at), mx[a] = lane_value(amx[a], at);
    }
    const int jy = b.mx[1] - b.mn[1], rows = jy * (b.mx[2] - b.mn[2]);
    for (int r = lane; r < rows; r += 64) set_cubes(keep_row(F, b.mn[1] + r % jy, b.mn[2] + r / jy), b.mn[0], b.mx[0]);
}

// Rows of a wave's common block whose cubes are gathered in LDS.
constexpr int LEAF_ROWS = 640;

// The leaves of paths [path0, path0 + npath) (path0 a multiple of 64), a lane
// each; a wave's 64 leaves share the block 6 halvings up, which is asked first,
// and whose cubes are gathered row by row before they go out.  The leaves left
// open go to the list, which holds npath.
__global__ __launch_bounds__(256) void k_filter_leaves(BlockFilter F, FBlock root, int depth, uint64_t path0,
                                                       uint64_t npath, uint64_t *__restrict__ open,
                                                       uint32_t *__restrict__ nopen) {
    __shared__ unsigned long long rows_all[4][LEAF_ROWS];
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // (scalar: so is the walk to the common block)
    unsigned long long *rows = rows_all[wid];
    const uint64_t wave = blockIdx.x * 4ull + wid, nw = gridDim.x * 4ull;
    const int above = depth > 6 ? depth - 6 : 0;
    for (uint64_t base = path0 + wave * 64; base < path0 + npath; base += nw * 64) {
        FBlock b = root;
        int d = 0;
        for (; d < above && !is_leaf(b); d++) halve(b, (base >> (depth - 1 - d)) & 1);
        double mn[3], mx[3];
        block_rect(F, b, mn, mx);
        const bool single = d < above;  // a leaf this far up: its first path stands for it
        if ((single && (base & ((1ull << (depth - d)) - 1))) || sure_miss(F.R, mn, mx)) continue;
        const uint64_t path = base + lane;
        FBlock l = b;
        bool valid = path < path0 + npath && (!single || lane == 0);
        if (!single) {
            for (; d < depth && !is_leaf(l); d++) halve(l, (path >> (depth - 1 - d)) & 1);
            valid = valid && (path & ((1ull << (depth - d)) - 1)) == 0;
        }
        bool acc = false, ask = false;
        if (valid) {
            block_rect(F, l, mn, mx);
            if (!sure_miss(F.R, mn, mx)) acc = sure_hit(F.R, mn, mx), ask = !acc;
        }
        const uint64_t am = __ballot(ask);
        if (am) {
            uint32_t at = 0;
            if (lane == 0) at = atomicAdd(nopen, (uint32_t)__popcll(am));
            at = lane_value(at, 0);
            if (ask) open[at + (uint32_t)__popcll(am & ((1ull << lane) - 1))] = path;
        }
        if (!__ballot(acc)) continue;
        const int bx = b.mx[0] - b.mn[0], by = b.mx[1] - b.mn[1], nrows = by * (b.mx[2] - b.mn[2]);
        const int jy = l.mx[1] - l.mn[1], lrows = acc ? jy * (l.mx[2] - l.mn[2]) : 0;
        if (nrows <= LEAF_ROWS && bx <= 64) {
            for (int r = lane; r < nrows; r += 64) rows[r] = 0;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const int lx = l.mx[0] - l.mn[0];
            const uint64_t m = (lx >= 64 ? ~0ull : ((1ull << lx) - 1)) << (l.mn[0] - b.mn[0]);
            for (int r = 0; r < lrows; r++)
                atomicOr(&rows[(l.mn[2] + r / jy - b.mn[2]) * by + (l.mn[1] + r % jy - b.mn[1])], (unsigned long long)m);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const int w = b.mn[0] >> 6, sh = b.mn[0] & 63;
            for (int r = lane; r < nrows; r += 64) {
                const uint64_t v = rows[r];
                if (!v) continue;
                unsigned long long *row = keep_row(F, b.mn[1] + r % by, b.mn[2] + r / by);
                atomicOr(&row[w], (unsigned long long)(v << sh));
                if (sh && (v >> (64 - sh))) atomicOr(&row[w + 1], (unsigned long long)(v >> (64 - sh)));
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        } else {
            for (int r = 0; r < lrows; r++) set_cubes(keep_row(F, l.mn[1] + r % jy, l.mn[2] + r / jy), l.mn[0], l.mx[0]);
        }
    }
}

__global__ __launch_bounds__(256) void k_filter_open(BlockFilter F, FBlock root, int depth,
                                                     const uint64_t *__restrict__ open,
                                                     const uint32_t *__restrict__ nopen) {
    const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, nw = (gridDim.x * blockDim.x) >> 6;
    const uint32_t n = *nopen;
    for (uint32_t i = wave; i < n; i += nw) open_leaf(F, root, depth, open[i]);
}

}  // namespace

hipError_t launch_rgrid_gather(const double *verts, const uint32_t *tris, uint64_t nt, double *out, hipStream_t st) {
    if (!nt) return hipSuccess;
    k_rgrid_gather<<<grid_for(9 * nt, 256, 4096), 256, 0, st>>>(verts, tris, nt, out);
    return hipGetLastError();
}

hipError_t launch_rgrid_count(const RectGridDev &R, GroupBox *box, uint32_t *counts, hipStream_t st) {
    if (!R.ntris) return hipSuccess;
    k_rgrid_count<<<grid_for(R.ntris, 256, 4096), 256, 0, st>>>(R, box, counts);
    return hipGetLastError();
}

hipError_t launch_rgrid_scan(const uint32_t *counts, uint32_t ncell, uint32_t *tiles, uint32_t *start,
                             uint32_t *cursor, hipStream_t st) {
    const uint32_t ntiles = (ncell + RSCAN - 1) / RSCAN;
    if (ncell == 0 || ntiles > RSCAN) return hipErrorInvalidValue;
    k_rscan_tiles<<<ntiles, RSCAN, 0, st>>>(counts, ncell, tiles);
    k_rscan_top<<<1, RSCAN, 0, st>>>(tiles, ntiles);
    k_rscan_down<<<ntiles, RSCAN, 0, st>>>(counts, ncell, tiles, start, cursor);
    return hipGetLastError();
}

hipError_t launch_rgrid_fill(const RectGridDev &R, uint32_t *cursor, uint32_t *cell_tris, hipStream_t st) {
    if (!R.ntris) return hipSuccess;
    k_rgrid_fill<<<grid_for(R.ntris, 256, 4096), 256, 0, st>>>(R, cursor, cell_tris);
    return hipGetLastError();
}

hipError_t launch_vgrid(const RectGridDev &R, uint32_t *vsat, hipStream_t st) {
    if (R.ntris) k_vgrid_count<<<grid_for(R.ntris, 256, 4096), 256, 0, st>>>(R, vsat);
    return launch_table(vsat, R.vn, st);
}

hipError_t launch_table(uint32_t *t, const int *n, hipStream_t st) {
    const uint32_t rows = (uint32_t)n[1] * n[2];
    k_vsat_x<<<grid_for(rows, 4, 4096), 256, 0, st>>>(t, n[0], rows);
    k_vsat_yz<<<grid_for((uint64_t)n[0] * n[2], 64, 4096), 64, 0, st>>>(t, n[0], n[1], n[2], 1);
    k_vsat_yz<<<grid_for((uint64_t)n[0] * n[1], 64, 4096), 64, 0, st>>>(t, n[0], n[1], n[2], 2);
    return hipGetLastError();
}

hipError_t launch_block_filter(const BlockFilter &F, const FBlock &root, int depth, uint64_t *open, uint32_t *nopen,
                               uint32_t ocap, hipStream_t st) {
    const uint64_t npath = 1ull << depth, part = std::min<uint64_t>(npath, ocap);
    for (uint64_t path0 = 0; path0 < npath; path0 += part) {
        const hipError_t e = launch_zero(nopen, 16, st);
        if (e != hipSuccess) return e;
        k_filter_leaves<<<grid_for(part, 256, 1u << 16), 256, 0, st>>>(F, root, depth, path0, part, open, nopen);
        k_filter_open<<<grid_for(part, 4, 2048), 256, 0, st>>>(F, root, depth, open, nopen);
    }
    return hipGetLastError();
}

}  // namespace mc3d
