// device.hpp -- device-side helpers shared by the kernels.
#pragma once

#include <algorithm>

#include <hip/hip_runtime.h>

namespace sodhip {

// Workgroup barrier for data exchanged through LDS by ordinary LDS stores:
// the wave's own LDS operations complete (lgkmcnt), then all waves meet.  The
// asm is a compiler barrier for memory accesses.  Neither __syncthreads nor a
// workgroup fence on LDS is used: the former also waits for every
// outstanding global load, the latter for every direct-to-LDS copy in flight,
// which would drain the prefetch of the next elements.  Data written by
// direct-to-LDS copies is read only after an explicit vmcnt wait.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// s_waitcnt immediate of vmcnt(0) (gfx9 encoding: vmcnt[3:0] | expcnt[6:4] |
// lgkmcnt[11:8] | vmcnt[5:4] << 14)
constexpr int kWaitVm0 = 0x0F70;

// Element order of the lane-per-node element loops: the blocks of one XCD
// (blockIdx % 8; the grid is a multiple of 8) walk one contiguous eighth of
// the elements, so elements that share cache lines (neighbouring nodes, the
// 16 elements of an element-fastest (nelem, nnode) line) run on one XCD and
// its L2.
struct XcdElems {
    int first, end, stride;
};
__device__ __forceinline__ XcdElems xcd_elems(int nelem)
{
    const int per = gridDim.x >> 3, xcd = blockIdx.x & 7, rk = blockIdx.x >> 3;
    const int span = (nelem + 7) >> 3;
    const int b = xcd * span;
    return {b + rk, min(nelem, b + span), per};
}

// Node order of the per-element reductions and limiters: alex[l] is the node at
// lexicographic position l of the element's (i, j, k) line indices (the inverse
// of the mesh cache's perm), so that a group of P+1 consecutive positions is one
// i-line: nodes that lie next to each other in memory on a structured numbering,
// read while their lines are still cached.  Built per block in LDS (nnode <= 125).
__device__ __forceinline__ void build_alex(const int *__restrict__ perm, int nnode, int *alex)
{
    for (int a = threadIdx.x; a < nnode; a += blockDim.x) alex[min(max(perm[a], 0), nnode - 1)] = a;
    __syncthreads();
}

// Those kernels read the reference's element-fastest (nelem, nnode) arrays.  A
// block of 256 threads takes tiles of 16 consecutive elements (whole 128-byte
// lines of an FP64 array): thread t holds element t % 16 and every 16th i-line from
// t / 16 on, one line at p=2 and p=3 and at most two at p=4.  (A thread per element
// walked all its lines one after the other, and a mesh of 1,728 elements
// occupied 7 of 256 CUs: 85 us for smart_visc_spectral_imex, now 11; at 41k elements
// 119 us, now 92.)  Each XCD takes one
// contiguous eighth of the tiles, whose shared nodes then sit in its L2.  The kernels
// are instances per line length KA: with five nodes read per line at every order, the
// index clamped, the tiles were slower than a thread per element on large meshes
// (343k elements, p=2: CFL step 97 us per thread, 127 clamped, 82 now; 262k, p=3: 200,
// 236 and 208 us; smart_visc_spectral_imex 142, 164, 124 and 232, 280, 224 us).
// The CFL step and the Ducros limit, which keep nothing between a tile's passes over
// memory, take tiles of W = 64 on meshes with two of those per CU: on large ones the
// 128-byte pieces of rows far apart cost more than the shorter walk gains, most where
// the row length is a power of two (calls, us, per thread / 16 / 64 wide: Ducros 262k
// elements, p=3: 274, 296, 256; 343k, p=2: 131, 121, 109; 41k, p=4: 149, 102, 98; CFL
// 221, 222, 183; 108, 90, 74; 92, 76, 70).  Smaller ones would idle CUs (8,000, p=4:
// Ducros 20 and 27 us, CFL 30 and 36 us, 16 and 64 wide).
constexpr int kTile = 16, kWideTile = 64;
inline bool wide_tiles(int nelem, int num_cu) { return nelem / kWideTile >= 2 * num_cu; }
// launches the kernel for KA = porder + 1 nodes per line (porder checked before)
#define SODHIP_BY_LINE(porder, launch, ...)                                                \
    do {                                                                                   \
        if ((porder) == 2) launch(3, ##__VA_ARGS__);                                       \
        else if ((porder) == 3) launch(4, ##__VA_ARGS__);                                  \
        else launch(5, ##__VA_ARGS__);                                                     \
    } while (0)
struct TileRange {
    int first, end, stride; // tiles
};
template <int W = kTile> __device__ __forceinline__ TileRange tile_range(int nelem)
{
    const int tiles = (nelem + W - 1) / W, span = (tiles + 7) >> 3;
    const int b = (blockIdx.x & 7) * span;
    return {b + (int)(blockIdx.x >> 3), min(tiles, b + span), (int)(gridDim.x >> 3)};
}
// at most eight blocks per CU
inline int tile_grid(int nelem, int num_cu, int width = kTile)
{
    const int tiles = (nelem + width - 1) / width, span = (tiles + 7) / 8;
    return 8 * std::max(1, std::min(span, num_cu));
}
// maximum over the 256 / W threads of each element; every thread returns its
// element's (sh: 4 W doubles)
template <int W = kTile> __device__ __forceinline__ double tile_max(double v, double *sh)
{
#pragma unroll
    for (int s = W; s < 64; s *= 2) v = fmax(v, __shfl_xor(v, s, 64));
    const int el = threadIdx.x % W;
    if ((threadIdx.x & 63) < W) sh[(threadIdx.x >> 6) * W + el] = v;
    __syncthreads();
    const double m = fmax(fmax(sh[el], sh[W + el]), fmax(sh[2 * W + el], sh[3 * W + el]));
    __syncthreads();
    return m;
}

} // namespace sodhip
