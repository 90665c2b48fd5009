// k_slab.hip -- stitching the meshes of a grid searched in z slabs.
//
// Slab s evaluates corner planes [z0, z1] and owns the cubes between; the
// plane z1 is also slab s + 1's first plane.  Each slab's search emits a
// vertex for every crossed edge its cubes use, so the x and y edges of a
// shared plane come out of both slabs, bit-identical (the same two corners
// and the same bisection).  The stitch keeps the lower slab's copy: the
// upper slab's copies are dropped and its triangles pointed at the lower
// slab's vertices, matched by edge (axis, x, y).
//
// After each slab, while its vertex keys are there, every vertex gets its
// offset from the slab's first vertex in the stitched mesh, and the edges of
// its top plane go into a hash table that the next slab looks its bottom
// plane's up in: the top plane's vertices are the slab's own, so no slab
// waits for another's place in the mesh.  When the slabs' sizes are known,
// all vertices and all triangles are moved by one launch each.  A slab of
// 10^5 vertices is bound by its launches: with flags, library scans, sorts of
// both planes' lists and the moves a slab at a time, seven slabs of a 512-atom
// solid at spacing 0.003 took 0.9 ms of kernels in 170 launches and two waits
// of the host a slab; now 0.2 ms in 16, and one wait in all.
#include "launch.h"

namespace mc3d {
namespace {

constexpr uint64_t KEY_XYA = (1ull << 42) - 1;  // a vertex key without its z (axis | x << 2 | y << 22)
constexpr uint64_t NO_KEY = ~0ull;

__device__ __forceinline__ bool on_plane(uint64_t key, int z) {
    return (key & 3) < 2 && (int)(key >> 42) == z;
}

// Vertices of a tile: SLAB_ITEMS consecutive ones a thread.
constexpr int SLAB_ITEMS = 4, SLAB_TILE = 256 * SLAB_ITEMS;
// Up to this many tiles a tile adds up the counts before it itself; more are
// scanned first.  (A tile's own sum reads at most 8 KB, eight loads a thread;
// a launch costs about 4 us.)
constexpr uint32_t SLAB_SUM_TILES = 2048;

__device__ __forceinline__ uint32_t slab_wave_inclusive(uint32_t v) {
    const int lane = threadIdx.x & 63;
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(v, d, 64);
        if (lane >= d) v += t;
    }
    return v;
}

// Edge (axis, x, y) of a table of 2^bits slots -> its first slot.
__device__ __forceinline__ uint64_t first_slot(uint64_t key, int bits) {
    return (key * 0x9e3779b97f4a7c15ull) >> (64 - bits);
}

// The bottom plane's vertices of every tile; the slab's table emptied.
__global__ __launch_bounds__(256) void k_slab_count(SlabPart S) {
    __shared__ uint32_t sh[4];
    if (blockIdx.x == 0 && threadIdx.x == 0) *S.end = SlabEnd{0, 0, 0, 0};
    if (S.ztop >= 0)
        for (uint64_t i = blockIdx.x * 256ull + threadIdx.x; i < (1ull << S.top_bits); i += gridDim.x * 256ull)
            S.top_keys[i] = NO_KEY;
    if (S.zbot < 0) return;
    for (uint32_t t = blockIdx.x; t < S.ntiles; t += gridDim.x) {
        uint32_t c = 0;
        for (int i = 0; i < SLAB_ITEMS; i++) {
            const uint64_t v = (uint64_t)t * SLAB_TILE + (uint64_t)i * 256 + threadIdx.x;
            c += (uint32_t)__popcll(__ballot(v < S.nv && on_plane(S.vkeys[v], S.zbot)));
        }
        __syncthreads();
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = c;
        __syncthreads();
        if (threadIdx.x == 0) S.counts[t] = sh[0] + sh[1] + sh[2] + sh[3];
    }
}

// Exclusive scan of the tiles' counts in place (one block).
__global__ __launch_bounds__(1024) void k_slab_scan(SlabPart S) {
    __shared__ uint32_t sh[16];
    uint32_t carry = 0;
    for (uint32_t t0 = 0; t0 < S.ntiles; t0 += 1024) {
        const uint32_t t = t0 + threadIdx.x, v = t < S.ntiles ? S.counts[t] : 0u;
        const uint32_t inc = slab_wave_inclusive(v);
        __syncthreads();
        if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6] = inc;
        __syncthreads();
        uint32_t pre = carry, all = 0;
        for (int w = 0; w < 16; w++) pre += w < (int)(threadIdx.x >> 6) ? sh[w] : 0u, all += sh[w];
        if (t < S.ntiles) S.counts[t] = pre + inc - v;
        carry += all;
    }
}

// rank[v]: the vertex's index in the stitched mesh less the slab's first
// (mod 2^32: a dropped vertex's copy lies before it).  Both tables have at
// most half their slots in use, so every probe ends at an empty one.
__global__ __launch_bounds__(256) void k_slab_rank(SlabPart S) {
    __shared__ uint32_t sh[4], sh_base[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t below = S.zbot >= 0 ? S.below_end->kept : 0u;
    for (uint32_t t = blockIdx.x; t < S.ntiles; t += gridDim.x) {
        uint64_t key[SLAB_ITEMS];
        const uint64_t v0 = (uint64_t)t * SLAB_TILE + threadIdx.x * SLAB_ITEMS;
        uint32_t sum = 0, tops = 0, bad = 0;
        for (int i = 0; i < SLAB_ITEMS; i++) key[i] = v0 + i < S.nv ? S.vkeys[v0 + i] : NO_KEY;
        for (int i = 0; i < SLAB_ITEMS; i++) sum += on_plane(key[i], S.zbot);  // (NO_KEY is on no plane)
        uint32_t base = 0;
        if (S.zbot >= 0) {
            if (S.scanned) {
                base = S.counts[t];
            } else {
                for (uint32_t i = threadIdx.x; i < t; i += 256) base += S.counts[i];
                for (int d = 32; d; d >>= 1) base += __shfl_xor(base, d, 64);
                if (lane == 0) sh_base[wave] = base;
            }
        }
        const uint32_t inc = slab_wave_inclusive(sum);
        if (lane == 63) sh[wave] = inc;
        __syncthreads();
        if (S.zbot >= 0 && !S.scanned) base = sh_base[0] + sh_base[1] + sh_base[2] + sh_base[3];
        for (int w = 0; w < wave; w++) base += sh[w];
        uint32_t dropped = base + inc - sum;  // before v0
        for (int i = 0; i < SLAB_ITEMS; i++) {
            if (v0 + i >= S.nv) break;
            const uint64_t edge = key[i] & KEY_XYA;
            uint32_t r = (uint32_t)(v0 + i) - dropped;
            if (on_plane(key[i], S.zbot)) {
                uint64_t s = first_slot(edge, S.below_bits), k;
                while ((k = S.below_keys[s]) != edge && k != NO_KEY) s = (s + 1) & ((1ull << S.below_bits) - 1);
                if (k == edge) r = S.below_vals[s] - below;
                else bad = 1;
                dropped++;
            } else if (on_plane(key[i], S.ztop)) {
                uint64_t s = first_slot(edge, S.top_bits);
                while (atomicCAS((unsigned long long *)&S.top_keys[s], NO_KEY, edge) != NO_KEY)
                    s = (s + 1) & ((1ull << S.top_bits) - 1);
                S.top_vals[s] = r;
                tops++;
            }
            S.rank[v0 + i] = r;
        }
        // (the last tile's last thread has seen every dropped vertex)
        if (t == S.ntiles - 1 && threadIdx.x == 255) {
            S.end->bottom = dropped;
            S.end->kept = (uint32_t)S.nv - dropped;
        }
        for (int d = 32; d; d >>= 1) tops += __shfl_xor(tops, d, 64);
        if (lane == 0 && tops) atomicAdd(&S.end->top, tops);
        if (bad) atomicOr(&S.end->bad, 1u);
        __syncthreads();
    }
}

// Every slab's own vertices (and interior points) to their place: a wave
// takes 64 vertices, 64 coordinates at a time; blockIdx.y takes slabs.
__global__ __launch_bounds__(256) void k_stitch_verts(const StitchPiece *__restrict__ pieces, uint32_t npieces,
                                                      double *__restrict__ fv, double *__restrict__ fin) {
    const uint32_t lane = threadIdx.x & 63;
    for (uint32_t k = blockIdx.y; k < npieces; k += gridDim.y) {
        const StitchPiece P = pieces[k];
        for (uint64_t v0 = blockIdx.x * 256ull + (threadIdx.x & ~63u); v0 < P.nv; v0 += gridDim.x * 256ull) {
            double x[3], y[3];
            uint32_t o[3], c[3];
            bool mine[3];
            for (int j = 0; j < 3; j++) {
                const uint32_t e = (uint32_t)j * 64 + lane, q = e / 3;
                c[j] = e - 3 * q;
                mine[j] = v0 + q < P.nv;
                o[j] = mine[j] ? P.vbase + P.rank[v0 + q] : 0;
                mine[j] = mine[j] && o[j] >= P.vbase;  // (else the slab below has it)
                x[j] = mine[j] ? P.v[3 * v0 + e] : 0;
                if (fin) y[j] = mine[j] ? P.in[3 * v0 + e] : 0;
            }
            for (int j = 0; j < 3; j++) {
                if (!mine[j]) continue;
                const uint64_t at = 3 * (uint64_t)o[j] + c[j];
                fv[at] = x[j];
                if (fin) fin[at] = y[j];
            }
        }
    }
}

// The triangles' indices, STITCH_ITEMS a thread in flight.
constexpr int STITCH_ITEMS = 8;
__global__ __launch_bounds__(256) void k_stitch_tris(const StitchPiece *__restrict__ pieces, uint32_t npieces,
                                                     uint32_t *__restrict__ ft) {
    for (uint32_t k = blockIdx.y; k < npieces; k += gridDim.y) {
        const StitchPiece P = pieces[k];
        const uint64_t n = 3 * P.nt, step = gridDim.x * (256ull * STITCH_ITEMS);
        for (uint64_t i0 = blockIdx.x * (256ull * STITCH_ITEMS) + threadIdx.x; i0 < n; i0 += step) {
            uint32_t t[STITCH_ITEMS];
            for (int j = 0; j < STITCH_ITEMS; j++) t[j] = i0 + j * 256 < n ? P.t[i0 + j * 256] : 0u;
            for (int j = 0; j < STITCH_ITEMS; j++) t[j] = P.vbase + P.rank[t[j]];
            for (int j = 0; j < STITCH_ITEMS; j++)
                if (i0 + j * 256 < n) ft[3 * P.tbase + i0 + j * 256] = t[j];
        }
    }
}

}  // namespace

uint32_t slab_tiles(uint64_t nv) { return (uint32_t)std::max<uint64_t>(1, (nv + SLAB_TILE - 1) / SLAB_TILE); }

hipError_t launch_slab_rank(SlabPart S, hipStream_t st) {
    S.ntiles = slab_tiles(S.nv);
    S.scanned = S.ntiles > SLAB_SUM_TILES;
    const unsigned grid = std::min(S.ntiles, 8192u);
    k_slab_count<<<grid, 256, 0, st>>>(S);
    if (S.scanned && S.zbot >= 0) k_slab_scan<<<1, 1024, 0, st>>>(S);
    k_slab_rank<<<grid, 256, 0, st>>>(S);
    return hipGetLastError();
}

hipError_t launch_stitch(const StitchPiece *pieces, uint32_t npieces, uint64_t nv_max, uint64_t nt_max, double *fv,
                         double *fin, uint32_t *ft, hipStream_t st) {
    const unsigned y = std::min(npieces, 4096u);
    if (nv_max) k_stitch_verts<<<dim3(grid_for(nv_max, 256, 2048), y), 256, 0, st>>>(pieces, npieces, fv, fin);
    if (nt_max) k_stitch_tris<<<dim3(grid_for(3 * nt_max, 256 * STITCH_ITEMS, 2048), y), 256, 0, st>>>(pieces, npieces, ft);
    return hipGetLastError();
}

}  // namespace mc3d
