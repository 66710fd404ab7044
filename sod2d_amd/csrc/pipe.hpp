// pipe.hpp -- input pipeline of the lane-per-node element kernels.
//
// A workgroup evaluates one unit of NE elements at a time (two at p=2, whose
// 27 nodes would leave more than half of a wave idle; one at p=3 and p=4) and
// walks a tile's units (unit_range).  Lane L owns the node at position L
// of the unit in lexicographic (I fastest) line order, so that
//   * the four or five nodes of an i-line, neighbours in memory on a mesh
//     numbered along i, are read by consecutive lanes: one gather of a field
//     touches a quarter of the cache lines it touches in gmsh order;
//   * the other nodes of a lane's three GLL lines lie at LDS positions a fixed
//     stride apart, which 16 consecutive lanes read without bank conflicts.
//
// Geometry (He, then gpvol) is copied HBM -> LDS by direct-to-LDS loads, one
// unit ahead, in rows of 64 lanes x 16 bytes.  A unit whose He block does not
// start on a 16-byte boundary (odd units at p=4: 9000 bytes per element) is
// copied from the boundary before it; the lanes then read from that many bytes
// (GeoAt) past the start of the LDS copy.  Rows of 4-byte lanes serve arrays that do
// not start on a 16-byte boundary and the last unit, whose rounded-up copy
// would run past the end of the arrays.
#pragma once

#include <algorithm>

#include "common.hpp"
#include "device.hpp"
#include "element.hpp"

namespace sodhip {

// direct-to-LDS copy of W (4 or 16) bytes per lane from g to lds + W*lane
// (lds wave-uniform), issued outside the compiler's wait tracking
template <int W> __device__ __forceinline__ void dma_lds(const void *g, unsigned lds)
{
    const unsigned m = __builtin_amdgcn_readfirstlane(lds);
    if constexpr (W == 16)
        asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(m) : "memory");
    else
        asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(g), "{m0}"(m) : "memory");
}

// wait until at most N of this wave's vector-memory operations are outstanding.  What
// the copies write may be read right after it: the builtin is not relied on to keep the
// compiler's reads behind the wait.
template <int N> __device__ __forceinline__ void wait_vm()
{
    static_assert(N >= 0 && N <= 63, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | kWaitVm0 | ((N >> 4) << 14));
    asm volatile("" ::: "memory");
}

// this wave's LDS reads have returned: a copy may overwrite what they read
__device__ __forceinline__ void lds_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// the value is formed by here (the compiler may not move its computation further on)
template <typename U> __device__ __forceinline__ void pin(U &x) { asm volatile("" : "+v"(x)); }

// LDS address of a __shared__ array
template <typename U> __device__ __forceinline__ unsigned lds_addr(U *p)
{
    return (unsigned)(uintptr_t)(__attribute__((address_space(3))) U *)p;
}

constexpr int gcd16(int n) { return n % 16 == 0 ? 16 : (n % 8 == 0 ? 8 : 4); }

template <int P, typename T> struct EP {
    static constexpr int N1 = P + 1, NN = N1 * N1 * N1;
    static constexpr int NE = P == 2 ? 2 : 1;          // elements per unit
    static constexpr int NL = NE * NN;                 // nodes (active lanes) per unit
    static constexpr int NT = (NL + 63) / 64 * 64;     // threads
    static constexpr int NW = NT / 64;
    // Units of a workgroup, consecutive ones: they share cache lines (the nodes of
    // neighbouring elements, the element-fastest mu arrays) that one CU then reads
    // once.  Four waves at p=3 and p=4 (553k elements, p=3, FP64: convection 1.41 ->
    // 1.25 ms, viscous operator 1.85 -> 1.54 ms against one unit per workgroup); at
    // p=2, where a unit already holds two elements, one wave without barriers is
    // faster (152k elements, both operators: 164 us against 184 us).
    static constexpr int G = P == 2 ? 1 : 4 / NW, NTB = G * NT;
    static constexpr int HEB = 9 * NL * (int)sizeof(T), GVB = NL * (int)sizeof(T);
    // room for a copy that starts up to 12 bytes early
    static constexpr int HEA = (HEB + (HEB % 16 ? 12 : 0) + 15) / 16 * 16;
    static constexpr int GVA = (GVB + (GVB % 16 ? 12 : 0) + 15) / 16 * 16;
    static constexpr int ROWS16 = (HEA + GVA + 1023) / 1024, ROWS4 = (HEA + GVA + 255) / 256;
    static constexpr int GEO = ROWS16 * 1024 > ROWS4 * 256 ? ROWS16 * 1024 : ROWS4 * 256;
    // no unit starts off a boundary and none reads past its own end
    static constexpr bool ALIGNED = HEB % 16 == 0 && GVB % 16 == 0;
};

// blocks of a workgroup's waves meet; a block of one wave only needs its own
// LDS operations complete (and the compiler not to move accesses across)
template <int NW> __device__ __forceinline__ void unit_sync()
{
    if constexpr (NW == 1) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    } else {
        lds_barrier();
    }
}

// The units of a block.  Each XCD (blockIdx % 8) owns one contiguous eighth of
// the units, cut into tiles of wide*run: block r of a tile takes units r,
// r + wide, ... of it.  Blocks are dispatched in order, so the blocks resident
// on an XCD work on consecutive units at a time.
struct UnitRange {
    int begin, end, stride;
};
__device__ __forceinline__ UnitRange unit_range(int nunits, int run, int wide)
{
    const int chunk = (nunits + 7) >> 3, rk = blockIdx.x >> 3;
    const int b = (blockIdx.x & 7) * chunk, e = min(nunits, b + chunk);
    const int t = b + rk / wide * wide * run;
    return {t + rk % wide, min(e, t + wide * run), wide};
}

// The launch over nelem elements.  A tile is as wide as the XCD has CUs (four
// times that for blocks of one wave), and a block takes up to 16 groups of
// units, fewer where that would leave the chip with less than two rounds of
// blocks; bpc, the stage's elem_blocks_per_cu setting, divides it by bpc / 16.  At 553k
// elements, p=3, FP64 the convection takes 1.25 ms with 16 groups in tiles of 32
// blocks, 1.29 ms with tiles of 128 and 1.26 ms with 8 groups; at 63k elements,
// p=4, 336, 349 and 347 us.  (One grid-stride walk over 128 blocks per CU, which
// amortises a block's tables over fewer units and drifts apart, took 1.46 ms and
// 429 us.)
struct UnitShape {
    int run, wide, grid;
};
template <int P, typename T> inline UnitShape unit_shape(sodhip_ctx ctx, int nelem, int bpc = 16)
{
    using Q = EP<P, T>;
    const int nunits = (nelem + Q::NE - 1) / Q::NE, ngroups = (nunits + Q::G - 1) / Q::G;
    const int cus = ctx->num_cu >= 8 ? ctx->num_cu / 8 : 1, chunk = (ngroups + 7) / 8;
    const int waves = Q::NTB / 64, round = cus * (8 / waves);
    UnitShape s;
    s.run = chunk / (2 * round);
    s.run = s.run < 1 ? 1 : (s.run > 16 ? 16 : s.run);
    if (bpc != 16) s.run = std::min(std::max(s.run * 16 / bpc, 1), 64);
    s.wide = cus * (4 / waves);
    const int tile = s.run * s.wide;
    s.grid = 8 * ((chunk + tile - 1) / tile * s.wide);
    return s;
}

// Where the LDS copy of a unit's geometry starts: bytes before He and gpvol
struct GeoAt {
    int he, gv;
};

// copies unit's He and, with VOL, gpvol to geo (LDS address); the waves take alternate
// rows
template <int P, typename T, bool VOL = true>
__device__ __forceinline__ GeoAt geo_issue(const T *He, const T *gpvol, int nelem, int nunits,
                                           bool geo16, int unit, unsigned geo, int wl, int wv)
{
    using Q = EP<P, T>;
    constexpr int END = Q::HEA + (VOL ? Q::GVA : 0);
    constexpr int ROWS16 = (END + 1023) / 1024, ROWS4 = (END + 255) / 256;
    const size_t hb = (size_t)unit * Q::HEB, gb = (size_t)unit * Q::GVB;
    const unsigned char *he = (const unsigned char *)He + hb;
    // without VOL the lanes past the end of He read its last bytes again
    const unsigned char *gv = VOL ? (const unsigned char *)gpvol + gb : he;
    const bool last = unit == nunits - 1;
    const bool wide = geo16 && (!last || (Q::ALIGNED && nelem % Q::NE == 0));
    if (wide) {
        const GeoAt at{Q::ALIGNED ? 0 : (int)(hb & 15), Q::ALIGNED ? 0 : (int)(gb & 15)};
        he -= at.he;
        gv -= VOL ? at.gv : at.he;
#pragma unroll
        for (int r0 = 0; r0 < ROWS16; r0 += Q::NW) {
            const int r = r0 + wv, byte = r * 1024 + wl * 16;
            const unsigned char *src = byte < Q::HEA ? he + byte
                                                     : gv + (VOL ? min(byte - Q::HEA, Q::GVA - 16) : Q::HEA - 16);
            if (ROWS16 % Q::NW == 0 || r < ROWS16) dma_lds<16>(src, geo + r * 1024);
        }
        return at;
    }
    // bytes of this unit that exist
    const int ne = min(Q::NE, nelem - unit * Q::NE);
    const int hlim = ne * (Q::HEB / Q::NE) - 4, glim = ne * (Q::GVB / Q::NE) - 4;
#pragma unroll 1
    for (int r = wv; r < ROWS4; r += Q::NW) {
        const int byte = r * 256 + wl * 4;
        const unsigned char *src =
            byte < Q::HEA || !VOL ? he + min(byte, hlim) : gv + min(byte - Q::HEA, glim);
        dma_lds<4>(src, geo + r * 256);
    }
    return {0, 0};
}

// The lane's place in a unit and its three GLL lines.  d/dxi_k at the lane's
// point has the coefficient ds[k] on its own value and d[k][o] on the P other
// nodes of the line, at unit positions nb[k][o]; t[k][o] is the transposed
// coefficient dl(b,k,I_k(a)) of the weak divergence (TRANS).  Tables are the
// caller's; indices are clamped so that malformed ones cannot address outside
// the element's arrays.
template <int P, typename T, bool TRANS> struct LexLane {
    static constexpr int N1 = P + 1, NN = N1 * N1 * N1;
    int sub, a, rec; // element of the unit, node (caller's order), record position
    int nb[3][P];
    T ds[3], d[3][P], t[TRANS ? 3 : 1][P];
    __device__ __forceinline__ LexLane(int lane, const T *__restrict__ dl,
                                       const int *__restrict__ inv, const int *__restrict__ perm)
    {
        constexpr int NL = EP<P, T>::NL;
        // lanes without a node evaluate the unit's first one again
        const int l = lane < NL ? lane : 0;
        sub = l / NN;
        const int pos = l - sub * NN;
        const int own[3] = {pos % N1, pos / N1 % N1, pos / (N1 * N1)};
        const int stride[3] = {1, N1, N1 * N1};
        auto node = [&](int p) { return min(max(inv[p] - 1, 0), NN - 1); };
        a = node(pos);
        rec = lane < NL ? sub * NN + min(max(perm[a], 0), NN - 1) : lane;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            ds[k] = dl[a + NN * (k + 3 * own[k])];
#pragma unroll
            for (int o = 0; o < P; ++o) {
                const int m = o + (o >= own[k] ? 1 : 0);
                const int q = pos + (m - own[k]) * stride[k];
                nb[k][o] = sub * NN + q;
                d[k][o] = dl[a + NN * (k + 3 * m)];
                if constexpr (TRANS) t[k][o] = dl[node(q) + NN * (k + 3 * own[k])];
            }
        }
    }
};

// A unit's records of RW values per node, written to LDS densely in the record order
// (LexLane::rec), go to out (elements back to back) as whole vectors: read into
// registers, then stored SB contiguous bytes per lane.
template <int P, typename T, int RW> struct RecOut {
    using Q = EP<P, T>;
    static constexpr int SB = gcd16(RW * Q::NL * (int)sizeof(T)), CH = RW * Q::NL * (int)sizeof(T) / SB,
                         NC = (CH + Q::NT - 1) / Q::NT;
    using U4 = unsigned __attribute__((ext_vector_type(4)));
    using U2 = unsigned __attribute__((ext_vector_type(2)));
    using V = std::conditional_t<SB == 16, U4, std::conditional_t<SB == 8, U2, unsigned>>;
    static __device__ __forceinline__ void read(V (&v)[NC], const T *area, int lane)
    {
#pragma unroll
        for (int i = 0; i < NC; ++i) v[i] = ((const V *)area)[min(lane + i * Q::NT, CH - 1)];
    }
    static __device__ __forceinline__ void store(const V (&v)[NC], const T *area, T *out, int u,
                                                 int nelem, int lane)
    {
        V *o = (V *)(out + (size_t)u * RW * Q::NL);
        if (Q::NE == 1 || (u + 1) * Q::NE <= nelem) {
#pragma unroll
            for (int i = 0; i < NC; ++i)
                if (lane + i * Q::NT < CH) o[lane + i * Q::NT] = v[i];
        } else { // the odd last element of a unit of two
            for (int i = lane; i < RW * Q::NN; i += Q::NT) ((T *)o)[i] = area[i];
        }
    }
};

} // namespace sodhip
