// ops_sensor.hip -- entropy-viscosity sensor smart_visc_spectral
// (mod_entropy_viscosity.f90:14-111) with the intra-element 3x3x3 filter of
// init_filters (mod_filters.f90:15-55).
//
// The entropy normalisation (mean of eta over working nodes in FP64, then the
// maximum deviation) is a deterministic two-level reduction: every block of
// the first kernel sums a fixed slice in a fixed tree order; the second kernel
// re-reduces the partial sums in the same fixed order in every block (all
// blocks obtain the identical mean) and forms partial maxima; the element
// kernel folds the partial maxima (max is order independent).  No host
// synchronisation is needed between the three launches.
#include <algorithm>
#include <cfloat>

#include "common.hpp"
#include "device.hpp"
#include "pipe.hpp"
#include "sensor.hpp"

namespace sodhip {

constexpr int kRedThreads = 256;

template <typename T> __device__ __forceinline__ T block_sum(T v, T *sh)
{
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (t < s) sh[t] = sh[t] + sh[t + s];
        __syncthreads();
    }
    T r = sh[0];
    __syncthreads();
    return r;
}

template <typename T> __device__ __forceinline__ T block_max(T v, T *sh)
{
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (t < s) sh[t] = fmax(sh[t], sh[t + s]);
        __syncthreads();
    }
    T r = sh[0];
    __syncthreads();
    return r;
}

// Block-wide sum of eta over the lpoin_w positions [i0, i1).  Four strided
// values are loaded ahead and added in the order of the plain strided loop,
// so the partial sums do not depend on the unrolling.
template <typename T>
__device__ __forceinline__ double eta_slice_sum(const int *__restrict__ lpoin_w,
                                                const T *__restrict__ eta, int i0, int i1,
                                                double *sh)
{
    const int bs = blockDim.x;
    double s = 0.0;
    int i = i0 + threadIdx.x;
    for (; i + 3 * bs < i1; i += 4 * bs) {
        const int n0 = lpoin_w[i], n1 = lpoin_w[i + bs], n2 = lpoin_w[i + 2 * bs],
                  n3 = lpoin_w[i + 3 * bs];
        const double v0 = (double)eta[n0 - 1], v1 = (double)eta[n1 - 1],
                     v2 = (double)eta[n2 - 1], v3 = (double)eta[n3 - 1];
        s += v0;
        s += v1;
        s += v2;
        s += v3;
    }
    for (; i < i1; i += bs) s += (double)eta[lpoin_w[i] - 1];
    return block_sum(s, sh);
}

// Block-wide max |eta - mean| over the lpoin_w positions [i0, i1), with mean
// the sum of the nparts partial sums part[] (in a fixed order) over nw.
template <typename T>
__device__ __forceinline__ double eta_slice_maxdev(const int *__restrict__ lpoin_w,
                                                   const T *__restrict__ eta,
                                                   const double *__restrict__ part, int nparts,
                                                   int nw, int i0, int i1, double *sh)
{
    double s = 0.0;
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) s += part[i];
    const double mean = block_sum(s, sh) / (double)nw;
    const int bs = blockDim.x;
    double m = 0.0;
    int i = i0 + threadIdx.x;
    for (; i + 3 * bs < i1; i += 4 * bs) {
        const int n0 = lpoin_w[i], n1 = lpoin_w[i + bs], n2 = lpoin_w[i + 2 * bs],
                  n3 = lpoin_w[i + 3 * bs];
        const double v0 = (double)eta[n0 - 1], v1 = (double)eta[n1 - 1],
                     v2 = (double)eta[n2 - 1], v3 = (double)eta[n3 - 1];
        m = fmax(fmax(m, fabs(v0 - mean)), fabs(v1 - mean));
        m = fmax(fmax(m, fabs(v2 - mean)), fabs(v3 - mean));
    }
    for (; i < i1; i += bs) m = fmax(m, fabs((double)eta[lpoin_w[i] - 1] - mean));
    return block_max(m, sh);
}

// partial sums of eta over working nodes: block b owns a contiguous slice
// (FP64 sums for either storage type)
template <typename T>
__global__ __launch_bounds__(kRedThreads) void k_eta_sum(int npoin_w, const int *__restrict__ lpoin_w,
                                                         const T *__restrict__ eta,
                                                         double *__restrict__ part)
{
    __shared__ double sh[kRedThreads];
    const int per = (npoin_w + gridDim.x - 1) / gridDim.x;
    const int i0 = blockIdx.x * per, i1 = min(npoin_w, i0 + per);
    const double s = eta_slice_sum(lpoin_w, eta, i0, i1, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// every block: mean = (sum of partial sums)/npoin_w in a fixed order, then its
// slice's max |eta - mean|
template <typename T>
__global__ __launch_bounds__(kRedThreads) void k_eta_maxdev(int npoin_w,
                                                            const int *__restrict__ lpoin_w,
                                                            const T *__restrict__ eta,
                                                            const double *__restrict__ part,
                                                            int nparts, double *__restrict__ pmax)
{
    __shared__ double sh[kRedThreads];
    const int per = (npoin_w + gridDim.x - 1) / gridDim.x;
    const int i0 = blockIdx.x * per, i1 = min(npoin_w, i0 + per);
    const double m = eta_slice_maxdev(lpoin_w, eta, part, nparts, npoin_w, i0, i1, sh);
    if (threadIdx.x == 0) pmax[blockIdx.x] = m;
}

// The same two passes per instance of a joined mesh: instance i owns the
// lpoin_w positions wseg[i]..wseg[i+1]-1 and the blocks i*nb..i*nb+nb-1,
// which split its segment as nb blocks split a single mesh's list (so the
// partials, mean and maximum have the bits of the instance run alone).
template <typename T>
__global__ __launch_bounds__(kRedThreads) void k_eta_sum_seg(const int *__restrict__ wseg, int nb,
                                                             const int *__restrict__ lpoin_w,
                                                             const T *__restrict__ eta,
                                                             double *__restrict__ part)
{
    __shared__ double sh[kRedThreads];
    const int inst = blockIdx.x / nb, b = blockIdx.x % nb;
    const int w0 = wseg[inst], nw = wseg[inst + 1] - w0;
    const int per = (nw + nb - 1) / nb;
    const int i0 = w0 + b * per, i1 = min(w0 + nw, i0 + per);
    const double s = eta_slice_sum(lpoin_w, eta, i0, i1, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = s;
}

template <typename T>
__global__ __launch_bounds__(kRedThreads) void k_eta_maxdev_seg(const int *__restrict__ wseg,
                                                                int nb,
                                                                const int *__restrict__ lpoin_w,
                                                                const T *__restrict__ eta,
                                                                const double *__restrict__ part,
                                                                double *__restrict__ pmax)
{
    __shared__ double sh[kRedThreads];
    const int inst = blockIdx.x / nb, b = blockIdx.x % nb;
    const int w0 = wseg[inst], nw = wseg[inst + 1] - w0;
    const int per = (nw + nb - 1) / nb;
    const int i0 = w0 + b * per, i1 = min(w0 + nw, i0 + per);
    const double m = eta_slice_maxdev(lpoin_w, eta, part + (size_t)inst * nb, nb, nw, i0, i1, sh);
    if (threadIdx.x == 0) pmax[blockIdx.x] = m;
}

// per instance: the maximum of its nb partial maxima (any order gives the
// same maximum)
__global__ __launch_bounds__(64) void k_norm_seg(int nb, const double *__restrict__ pmax,
                                                 double *__restrict__ norm_i)
{
    double m = 0.0;
    for (int i = threadIdx.x; i < nb; i += 64) m = fmax(m, pmax[(size_t)blockIdx.x * nb + i]);
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) m = fmax(m, __shfl_xor(m, s, 64));
    if (threadIdx.x == 0) norm_i[blockIdx.x] = m;
}

template <typename T> __device__ __forceinline__ T block_min(T v, T *sh)
{
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (t < s) sh[t] = fmin(sh[t], sh[t + s]);
        __syncthreads();
    }
    T r = sh[0];
    __syncthreads();
    return r;
}

// partial minima of rho over working nodes (contiguous slices), starting
// from the reference's 100000
__global__ __launch_bounds__(kRedThreads) void k_rho_min(int npoin_w, const int *__restrict__ lpoin_w,
                                                         const double *__restrict__ rho,
                                                         double *__restrict__ part)
{
    __shared__ double sh[kRedThreads];
    const int per = (npoin_w + gridDim.x - 1) / gridDim.x;
    const int i0 = blockIdx.x * per, i1 = min(npoin_w, i0 + per);
    double m = 100000.0;
    for (int i = i0 + threadIdx.x; i < i1; i += blockDim.x) m = fmin(m, rho[lpoin_w[i] - 1]);
    m = block_min(m, sh);
    if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// smart_visc_spectral_imex (mod_entropy_viscosity.f90:113-227) over tiles of 16
// elements (device.hpp): mue_l <- incoming mu_e; beta_e = max over the nodes of rho helem_k (cmax/p)
// (|u| + fact c); mu_e = cglob min(ce rho |Reta|/norm (helem_k/p)^2, beta_e).
// norm: 1, or the max of the partials (max |eta - mean|), or the min of the
// partials (min rho), folded per block.  All loads of an i-line are issued
// together; density and residual stay in registers between the maximum and the
// write.
struct ImexArgs {
    int nelem, nnode, porder;
    const int *connec, *perm;
    const double *Reta, *rho, *u, *csound, *helem_k;
    int npoin;
    double ce, cmax, cglob, fact_low_mach;
    const double *part; // partials of the norm, or nullptr (norm = 1)
    int nparts, norm_min;
    double *mu_e, *mue_l;
};

template <int KA>
__global__ __launch_bounds__(256) void k_visc_imex(ImexArgs A)
{
    __shared__ double sh[256];
    __shared__ int alex[125];
    build_alex(A.perm, A.nnode, alex);
    double norm = 1.0;
    if (A.part) {
        double v = A.norm_min ? 100000.0 : 0.0;
        for (int i = threadIdx.x; i < A.nparts; i += blockDim.x)
            v = A.norm_min ? fmin(v, A.part[i]) : fmax(v, A.part[i]);
        norm = A.norm_min ? block_min(v, sh) : block_max(v, sh);
    }
    const size_t NE = (size_t)A.nelem;
    const double *u1 = A.u + A.npoin, *u2 = A.u + 2 * (size_t)A.npoin;
    const double cp = A.cmax / (double)A.porder;
    constexpr int nl = KA * KA, LINES = (nl + 15) / 16;
    const TileRange tr = tile_range(A.nelem);
    for (int t = tr.first; t < tr.end; t += tr.stride) {
        const int el = t * kTile + (threadIdx.x & 15), e = min(el, A.nelem - 1);
        const double hk = A.helem_k[e];
        double betae = 0.0;
        double rh[LINES][KA], re[LINES][KA];
#pragma unroll
        for (int r = 0; r < LINES; ++r) {
            const int l = (threadIdx.x >> 4) + 16 * r;
            if (l >= nl) break;
            size_t ea[KA];
            int n[KA];
            double mu[KA], v0[KA], v1[KA], v2[KA], cs[KA];
#pragma unroll
            for (int j = 0; j < KA; ++j) {
                ea[j] = e + NE * alex[l * KA + j];
                n[j] = A.connec[ea[j]] - 1;
                mu[j] = A.mu_e[ea[j]];
            }
#pragma unroll
            for (int j = 0; j < KA; ++j) {
                v0[j] = A.u[n[j]];
                v1[j] = u1[n[j]];
                v2[j] = u2[n[j]];
                cs[j] = A.csound[n[j]];
                rh[r][j] = A.rho[n[j]];
                re[r][j] = A.Reta[n[j]];
            }
#pragma unroll
            for (int j = 0; j < KA; ++j) {
                if (el < A.nelem) A.mue_l[ea[j]] = mu[j];
                const double speed =
                    sqrt(v0[j] * v0[j] + v1[j] * v1[j] + v2[j] * v2[j]) + A.fact_low_mach * cs[j];
                betae = fmax(betae, (rh[r][j] * hk) * cp * speed);
            }
        }
        betae = tile_max(betae, sh);
        if (el >= A.nelem) continue;
        const double hp = hk / (double)A.porder;
#pragma unroll
        for (int r = 0; r < LINES; ++r) {
            const int l = (threadIdx.x >> 4) + 16 * r;
            if (l >= nl) break;
#pragma unroll
            for (int j = 0; j < KA; ++j) {
                const double R1 = rh[r][j] * fabs(re[r][j]) / norm;
                const double Ve = A.ce * R1 * (hp * hp);
                A.mu_e[e + NE * alex[l * KA + j]] = A.cglob * fmin(Ve, betae);
            }
        }
    }
}

// ducros_visc_limit (mod_entropy_viscosity.f90:277-314) in two passes.  Of
// the limiter's inputs only helem and mu_e are per element-node; the rest
// depends on the node alone.  A node pass forms, per node, d2 = (divU/Ml)^2,
// phi = min(4/3 d2 / (d2 + |curl u|^2 + eps), 1) and |u| (three arrays, read
// and written in streams); the element pass gathers those three instead of
// the eight node fields (eight gather streams per node overran the caches:
// about 3.7 times the algorithmic bytes were fetched).  Same expressions,
// same bits as one pass.
__global__ __launch_bounds__(256) void k_ducros_node(int npoin, const double *__restrict__ u,
                                                     const double *__restrict__ divU,
                                                     const double *__restrict__ vorti,
                                                     const double *__restrict__ Ml,
                                                     double *__restrict__ nq)
{
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= npoin) return;
    const size_t P1 = (size_t)npoin, P2 = 2 * (size_t)npoin;
    const double dv = divU[n] / Ml[n];
    const double w0 = vorti[n], w1 = vorti[n + P1], w2 = vorti[n + P2];
    const double v0 = u[n], v1 = u[n + P1], v2 = u[n + P2];
    const double d2 = dv * dv;
    nq[n] = fmin((4.0 / 3.0) * d2 / (d2 + (w0 * w0 + w1 * w1 + w2 * w2) + DBL_EPSILON), 1.0);
    nq[n + P1] = d2;
    nq[n + P2] = sqrt(v0 * v0 + v1 * v1 + v2 * v2);
}

// the element pass, over tiles of W elements (device.hpp), all loads of an i-line
// issued together
template <int KA, int W>
__global__ __launch_bounds__(256) void k_ducros(int nelem, int nnode, int porder, int npoin,
                                                const int *__restrict__ connec,
                                                const int *__restrict__ perm,
                                                const double *__restrict__ nq,
                                                const double *__restrict__ helem, double dmin,
                                                double *__restrict__ mu_e)
{
    __shared__ int alex[125];
    build_alex(perm, nnode, alex);
    const size_t P1 = (size_t)npoin, P2 = 2 * (size_t)npoin;
    constexpr int nl = KA * KA;
    const TileRange tr = tile_range<W>(nelem);
    for (int tile = tr.first; tile < tr.end; tile += tr.stride) {
        const int e = tile * W + threadIdx.x % W;
        if (e >= nelem) continue;
        for (int l = threadIdx.x / W; l < nl; l += 256 / W) {
            size_t t[KA];
            int n[KA];
#pragma unroll
            for (int j = 0; j < KA; ++j) {
                t[j] = (size_t)alex[l * KA + j] * nelem + e;
                n[j] = connec[t[j]] - 1;
            }
            double phi[KA], d2[KA], um[KA], he[KA], mu[KA];
#pragma unroll
            for (int j = 0; j < KA; ++j) {
                phi[j] = nq[n[j]];
                d2[j] = nq[n[j] + P1];
                um[j] = nq[n[j] + P2];
                he[j] = helem[t[j]];
                mu[j] = mu_e[t[j]];
            }
#pragma unroll
            for (int j = 0; j < KA; ++j) {
                const double rr = 1.0 * um[j] / he[j];
                const double phi2 = d2[j] / (d2[j] + rr * rr + DBL_EPSILON);
                mu_e[t[j]] = mu[j] * (fmax(phi[j] - dmin, 0.0) * phi2 + dmin);
            }
        }
    }
}

// max over each row of 16 lanes, by DPP rotations
__device__ __forceinline__ double row_max(double v)
{
    auto ror = [](double x, auto n) {
        constexpr int ctrl = 0x120 + decltype(n)::value;
        const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(x), ctrl, 0xf, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(x), ctrl, 0xf, 0xf, false);
        return __hiloint2double(hi, lo);
    };
    v = fmax(v, ror(v, std::integral_constant<int, 8>{}));
    v = fmax(v, ror(v, std::integral_constant<int, 4>{}));
    v = fmax(v, ror(v, std::integral_constant<int, 2>{}));
    return fmax(v, ror(v, std::integral_constant<int, 1>{}));
}
// ... and over the wave
__device__ __forceinline__ double wave_max(double v)
{
    v = row_max(v);
    v = fmax(v, __shfl_xor(v, 16, 64));
    return fmax(v, __shfl_xor(v, 32, 64));
}

// smart_visc_spectral over chunks of CH = 16 consecutive elements, so that the
// element-fastest arrays helem(nelem,nnode), mue_l and mu_e move as whole 128-byte
// lines through LDS (thread t holds node t/CH of element t%CH).  In between, lanes
// hold nodes in line order (I fastest), as the operators' kernels do: a gather then
// touches a quarter of the cache lines that it touches in gmsh order.  Groups of NT
// lanes (one wave; two at p=4) take NE elements at a time (two at p=2), and every
// group's share of the chunk, E rounds, is in flight at once.
//
// What bounds it: waits on L2 for the gathers of six node fields (the vector memory
// units stall on lines in flight 0.7 of the time, whatever the occupancy).  48 bytes
// per element-node and the node fields once would take 145 us of a large copy's rate at
// 262k elements, p=3; it takes 284 us, 404 with one wave per chunk in gmsh order, which
// also read the filter's 27 sources one by one and rows of 64 doubles whose 16
// elements share a bank pair.  48k elements, p=4: 167 -> 131 us; 152k, p=2: 155 -> 68 us;
// 512 elements, p=3 (32 waves): 28 -> 8.5 us.  The filter is three line passes of two
// LDS reads, and rows are padded to an odd number of doubles.
template <int P> struct SensorShape {
    static constexpr int NN = SG<P>::NN, NT = SG<P>::NT, NW = NT / 64, CH = 16;
    static constexpr int NE = P == 2 ? 2 : 1, G = 4, NTB = G * NT; // groups, threads
    static constexpr int E = CH / (G * NE), ROW = NN | 1;
};

template <int P, typename S>
__global__ __launch_bounds__(SensorShape<P>::NTB, 4) void k_smart_visc(SensorArgsT<S> A)
{
    using Q = SensorShape<P>;
    constexpr int NN = Q::NN, NT = Q::NT, NW = Q::NW, CH = Q::CH, NE = Q::NE, E = Q::E, ROW = Q::ROW;
    constexpr int BLK = CH * NN, ROWS = (BLK + Q::NTB - 1) / Q::NTB;
    __shared__ double lb[CH * ROW], ob[CH * ROW];
    __shared__ double wmax[NW > 1 ? Q::G * NW * E : 1];
    const int grp = threadIdx.x / NT, lane = threadIdx.x % NT, wl = threadIdx.x & 63;
    const bool act = lane < NE * NN;
    const int sub = act ? lane / NN : 0, at = act ? lane - sub * NN : 0;
    const int a = min(max(A.inv[at] - 1, 0), NN - 1);
    const FilterLane<P> fl(at);
    double norm = 1.0;
    if (A.pmax) { // every wave folds all partial maxima itself
        norm = 0.0;
        for (int i = wl; i < A.nparts; i += 64) norm = fmax(norm, A.pmax[i]);
        norm = wave_max(norm);
    }
    const size_t np = (size_t)A.npoin;
    const TileRange tr = tile_range(A.nelem);
    if (tr.first >= tr.end) return;
    // element of round r in the chunk, and its place in LDS
    auto slot = [&](int r) { return (r * Q::G + grp) * NE + sub; };
    auto elem = [&](int tile, int r) { return min(tile * CH + slot(r), A.nelem - 1); };
    int n[E];
#pragma unroll
    for (int r = 0; r < E; ++r) n[r] = A.connecT[(size_t)elem(tr.first, r) * NN + a];
    for (int tile = tr.first; tile < tr.end; tile += tr.stride) {
        const int c0 = tile * CH, cn = min(CH, A.nelem - c0);
        double u0[E], u1[E], u2[E], T[E], rho[E], re[E], hk[E];
#pragma unroll
        for (int r = 0; r < E; ++r) {
            u0[r] = A.u[n[r]];
            u1[r] = A.u[n[r] + np];
            u2[r] = A.u[n[r] + 2 * np];
            T[r] = A.Tem[n[r]];
            rho[r] = A.rho[n[r]];
            re[r] = A.Reta[n[r]];
            hk[r] = A.helem_k[elem(tile, r)];
        }
        // helem of the chunk (elements past the last re-read it)
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int t = i * Q::NTB + threadIdx.x;
            if (t < BLK) lb[t % CH * ROW + t / CH] = A.helem[c0 + min(t % CH, cn - 1) + (size_t)A.nelem * (t / CH)];
        }
        const int tnext = tile + tr.stride < tr.end ? tile + tr.stride : tile;
#pragma unroll
        for (int r = 0; r < E; ++r) n[r] = A.connecT[(size_t)elem(tnext, r) * NN + a];
        double be[E];
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const double aux2 = sqrt(u0[r] * u0[r] + u1[r] * u1[r] + u2[r] * u2[r]);
            const double aux3 = A.fact_low_mach * sqrt(A.Rgas * A.gamma * T[r]);
            const double b = act ? (rho[r] * hk[r]) * (A.cmax / (double)P) * (aux2 + aux3) : 0.0;
            if constexpr (NE == 2) {
                const double b0 = wave_max(sub == 0 ? b : 0.0), b1 = wave_max(sub == 1 ? b : 0.0);
                be[r] = sub == 0 ? b0 : b1;
            } else {
                be[r] = wave_max(b);
                if constexpr (NW > 1)
                    if (wl == 0) wmax[(grp * NW + lane / 64) * E + r] = be[r];
            }
        }
        lds_barrier();
        double ml[E];
#pragma unroll
        for (int r = 0; r < E; ++r) {
            if constexpr (NW > 1) {
#pragma unroll
                for (int w = 0; w < NW; ++w) be[r] = fmax(be[r], wmax[(grp * NW + w) * E + r]);
            }
            const double nrm = A.norm_i ? A.norm_i[A.elem_inst[elem(tile, r)]] : norm;
            const double R1 = rho[r] * fabs(re[r]) / nrm;
            const double h = lb[slot(r) * ROW + a];
            const double Ve = A.ce * R1 * (h * h);
            ml[r] = A.cglob * fmin(Ve, be[r]);
        }
        // the three line passes, lb -> ob -> lb, in line order (a group's own rows)
        double v[E];
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = ml[r];
        unit_sync<NW>();
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            double *const buf = k == 1 ? ob : lb;
            if (act)
#pragma unroll
                for (int r = 0; r < E; ++r) buf[slot(r) * ROW + at] = v[r];
            unit_sync<NW>();
#pragma unroll
            for (int r = 0; r < E; ++r)
                v[r] = filter_line(buf[slot(r) * ROW + fl.n[k][0]], v[r], buf[slot(r) * ROW + fl.n[k][1]]);
        }
        unit_sync<NW>();
        if (act)
#pragma unroll
            for (int r = 0; r < E; ++r) {
                lb[slot(r) * ROW + a] = ml[r];
                ob[slot(r) * ROW + a] = v[r];
            }
        lds_barrier();
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int t = i * Q::NTB + threadIdx.x;
            if (t < BLK && t % CH < cn) {
                const size_t g = c0 + t % CH + (size_t)A.nelem * (t / CH);
                A.mue_l[g] = lb[t % CH * ROW + t / CH];
                A.mu_e[g] = ob[t % CH * ROW + t / CH];
            }
        }
        lds_barrier(); // the next chunk overwrites lb and ob
    }
}

// The entropy normalisation's partial maxima of |eta - mean| over the working
// nodes (kRedBlocks values in ctx->scratch2), or nullptr when the sensor does
// not normalise; for kernels that fold them as the sensor does.
int entropy_norm_partials(sodhip_ctx ctx, int npoin_w, const int *lpoin_w, const double *eta,
                          bool normalise, const double **pmax, int *nparts)
{
    *pmax = nullptr;
    *nparts = kRedBlocks;
    if (!normalise) return SODHIP_OK;
    int rc = ensure_buf(ctx->scratch2, 2 * kRedBlocks * sizeof(double));
    if (rc) return rc;
    double *part = (double *)ctx->scratch2.ptr;
    k_eta_sum<double><<<kRedBlocks, kRedThreads, 0, ctx->stream>>>(npoin_w, lpoin_w, eta, part);
    k_eta_maxdev<double><<<kRedBlocks, kRedThreads, 0, ctx->stream>>>(npoin_w, lpoin_w, eta, part,
                                                              kRedBlocks, part + kRedBlocks);
    SODHIP_TRY_HIP(hipGetLastError());
    *pmax = part + kRedBlocks;
    return SODHIP_OK;
}

int entropy_norm_instances(sodhip_ctx ctx, const sodhip_instances *ens, const int *lpoin_w,
                           const double *eta, const double **norm_i)
{
    SODHIP_REQUIRE(ens && ens->ninst > 0 && ens->wseg && ens->elem_inst, "invalid instances");
    const size_t np = (size_t)ens->ninst * kRedBlocks;
    int rc = ensure_buf(ctx->scratch2, (2 * np + ens->ninst) * sizeof(double));
    if (rc) return rc;
    double *part = (double *)ctx->scratch2.ptr, *pmax = part + np, *nrm = pmax + np;
    const int grid = ens->ninst * kRedBlocks;
    k_eta_sum_seg<double><<<grid, kRedThreads, 0, ctx->stream>>>(ens->wseg, kRedBlocks, lpoin_w,
                                                                 eta, part);
    k_eta_maxdev_seg<double><<<grid, kRedThreads, 0, ctx->stream>>>(ens->wseg, kRedBlocks,
                                                                    lpoin_w, eta, part, pmax);
    k_norm_seg<<<ens->ninst, 64, 0, ctx->stream>>>(kRedBlocks, pmax, nrm);
    SODHIP_TRY_HIP(hipGetLastError());
    *norm_i = nrm;
    return SODHIP_OK;
}

} // namespace sodhip

using namespace sodhip;

template <typename T>
static int smart_visc(sodhip_ctx ctx, int porder, int nelem, int npoin, int npoin_w,
                      const int *connec, const int *lpoin_w, const T *Reta, double gamma_gas,
                      const T *rho, const T *u, const T *Tem, const T *eta, const T *helem,
                      const T *helem_k, const int *invAtoIJK, const sodhip_visc_params *prm,
                      T *mu_e, T *mue_l, const sodhip_instances *ens = nullptr)
{
    SODHIP_REQUIRE(ctx && prm, "null argument");
    SODHIP_REQUIRE(porder >= 2 && porder <= kMaxP, "porder %d not supported (2..4)", porder);
    SODHIP_REQUIRE(nelem > 0 && npoin > 0 && npoin_w > 0 && npoin_w <= npoin,
                   "invalid mesh sizes");
    SODHIP_REQUIRE(connec && lpoin_w && Reta && rho && u && Tem && eta && helem && helem_k &&
                       invAtoIJK && mu_e && mue_l,
                   "null array argument");
    SODHIP_TRY_HIP(hipSetDevice(ctx->device));
    MeshCache *m = nullptr;
    int rc = get_mesh(ctx, porder, nelem, npoin, connec, &m);
    if (rc) return rc;
    if ((rc = ensure_buf(ctx->scratch2, 2 * kRedBlocks * sizeof(double)))) return rc;
    double *part = (double *)ctx->scratch2.ptr;
    double *pmax = part + kRedBlocks;
    const bool normalise = prm->flag_normalise_entropy == 1;
    int tok = prof_begin(ctx, 2);
    const double *norm_i = nullptr;
    if (normalise && ens) {
        if constexpr (sizeof(T) == 8) {
            if ((rc = entropy_norm_instances(ctx, ens, lpoin_w, eta, &norm_i))) return rc;
        }
    } else if (normalise) {
        k_eta_sum<T><<<kRedBlocks, kRedThreads, 0, ctx->stream>>>(npoin_w, lpoin_w, eta, part);
        k_eta_maxdev<T><<<kRedBlocks, kRedThreads, 0, ctx->stream>>>(npoin_w, lpoin_w, eta, part,
                                                                     kRedBlocks, pmax);
    }
    SensorArgsT<T> A{};
    A.nelem = nelem;
    A.npoin = npoin;
    A.connecT = m->connecT;
    A.Reta = Reta;
    A.rho = rho;
    A.u = u;
    A.Tem = Tem;
    A.helem = helem;
    A.helem_k = helem_k;
    A.inv = invAtoIJK;
    A.gamma = gamma_gas;
    A.Rgas = prm->Rgas;
    A.ce = prm->ce;
    A.cmax = prm->cmax;
    A.cglob = prm->cglob;
    A.fact_low_mach = prm->flag_drop_c_in_envit ? 0.0 : 1.0;
    A.pmax = normalise && !ens ? pmax : nullptr;
    A.nparts = kRedBlocks;
    A.norm_i = norm_i;
    A.elem_inst = norm_i ? ens->elem_inst : nullptr;
    A.mu_e = mu_e;
    A.mue_l = mue_l;
    const int grid = tile_grid(nelem, ctx->num_cu);
    switch (porder) {
    case 2: k_smart_visc<2, T><<<grid, SensorShape<2>::NTB, 0, ctx->stream>>>(A); break;
    case 3: k_smart_visc<3, T><<<grid, SensorShape<3>::NTB, 0, ctx->stream>>>(A); break;
    case 4: k_smart_visc<4, T><<<grid, SensorShape<4>::NTB, 0, ctx->stream>>>(A); break;
    }
    prof_end(ctx, tok);
    SODHIP_TRY_HIP(hipGetLastError());
    return SODHIP_OK;
}

extern "C" int sodhip_smart_visc_spectral_f64(sodhip_ctx ctx, int porder, int nelem, int npoin,
                                              int npoin_w, const int *connec, const int *lpoin_w,
                                              const double *Reta, double gamma_gas,
                                              const double *rho, const double *u,
                                              const double *Tem, const double *eta,
                                              const double *helem, const double *helem_k,
                                              const int *invAtoIJK, const sodhip_visc_params *prm,
                                              double *mu_e, double *mue_l)
{
    return smart_visc<double>(ctx, porder, nelem, npoin, npoin_w, connec, lpoin_w, Reta, gamma_gas,
                              rho, u, Tem, eta, helem, helem_k, invAtoIJK, prm, mu_e, mue_l);
}

extern "C" int sodhip_smart_visc_spectral_ens_f64(
    sodhip_ctx ctx, int porder, int nelem, int npoin, int npoin_w, const int *connec,
    const int *lpoin_w, const sodhip_instances *ens, const double *Reta, double gamma_gas,
    const double *rho, const double *u, const double *Tem, const double *eta,
    const double *helem, const double *helem_k, const int *invAtoIJK,
    const sodhip_visc_params *prm, double *mu_e, double *mue_l)
{
    SODHIP_REQUIRE(ens && ens->ninst > 0 && ens->wseg && ens->elem_inst, "invalid instances");
    return smart_visc<double>(ctx, porder, nelem, npoin, npoin_w, connec, lpoin_w, Reta, gamma_gas,
                              rho, u, Tem, eta, helem, helem_k, invAtoIJK, prm, mu_e, mue_l, ens);
}

extern "C" int sodhip_smart_visc_spectral_f32(sodhip_ctx ctx, int porder, int nelem, int npoin,
                                              int npoin_w, const int *connec, const int *lpoin_w,
                                              const float *Reta, float gamma_gas,
                                              const float *rho, const float *u, const float *Tem,
                                              const float *eta, const float *helem,
                                              const float *helem_k, const int *invAtoIJK,
                                              const sodhip_visc_params *prm, float *mu_e,
                                              float *mue_l)
{
    return smart_visc<float>(ctx, porder, nelem, npoin, npoin_w, connec, lpoin_w, Reta,
                             (double)gamma_gas, rho, u, Tem, eta, helem, helem_k, invAtoIJK, prm,
                             mu_e, mue_l);
}

extern "C" int sodhip_smart_visc_spectral_imex_f64(
    sodhip_ctx ctx, int porder, int nelem, int npoin, int npoin_w, const int *connec,
    const int *lpoin_w, const double *Reta, const double *rho, const double *u,
    const double *csound, const double *eta, const double *helem_k, sodhip_visc_params *prm,
    double ce_comp, int flag_high_mach, double *mu_e, double *mue_l)
{
    SODHIP_REQUIRE(ctx && prm, "null argument");
    SODHIP_REQUIRE(porder >= 2 && porder <= kMaxP, "porder %d not supported (2..4)", porder);
    SODHIP_REQUIRE(nelem > 0 && npoin > 0 && npoin_w > 0 && npoin_w <= npoin,
                   "invalid mesh sizes");
    SODHIP_REQUIRE(connec && lpoin_w && Reta && rho && u && csound && eta && helem_k && mu_e &&
                       mue_l,
                   "null array argument");
    SODHIP_TRY_HIP(hipSetDevice(ctx->device));
    MeshCache *m = nullptr;
    int rc = get_mesh(ctx, porder, nelem, npoin, connec, &m);
    if (rc) return rc;
    if ((rc = ensure_buf(ctx->scratch2, 2 * kRedBlocks * sizeof(double)))) return rc;
    double *part = (double *)ctx->scratch2.ptr;
    double *pmax = part + kRedBlocks;
    const bool normalise = prm->flag_normalise_entropy == 1;
    const bool high_mach = normalise && flag_high_mach;
    int tok = prof_begin(ctx, 2);
    if (high_mach) {
        k_rho_min<<<kRedBlocks, kRedThreads, 0, ctx->stream>>>(npoin_w, lpoin_w, rho, pmax);
        // the reference assigns its module global ce (kept for later calls)
        prm->ce = ce_comp;
    } else if (normalise) {
        k_eta_sum<double><<<kRedBlocks, kRedThreads, 0, ctx->stream>>>(npoin_w, lpoin_w, eta, part);
        k_eta_maxdev<double><<<kRedBlocks, kRedThreads, 0, ctx->stream>>>(npoin_w, lpoin_w, eta, part,
                                                                  kRedBlocks, pmax);
    }
    ImexArgs A{};
    A.nelem = nelem;
    A.nnode = (porder + 1) * (porder + 1) * (porder + 1);
    A.porder = porder;
    A.connec = connec;
    A.perm = m->perm;
    A.Reta = Reta;
    A.rho = rho;
    A.u = u;
    A.csound = csound;
    A.helem_k = helem_k;
    A.npoin = npoin;
    A.ce = prm->ce;
    A.cmax = prm->cmax;
    A.cglob = prm->cglob;
    A.fact_low_mach = prm->flag_drop_c_in_envit ? 0.0 : 1.0;
    A.part = normalise ? pmax : nullptr;
    A.nparts = kRedBlocks;
    A.norm_min = high_mach ? 1 : 0;
    A.mu_e = mu_e;
    A.mue_l = mue_l;
#define SODHIP_IMEX(KA) \
    k_visc_imex<KA><<<tile_grid(nelem, ctx->num_cu), 256, 0, ctx->stream>>>( \
        A)
    SODHIP_BY_LINE(porder, SODHIP_IMEX);
#undef SODHIP_IMEX
    prof_end(ctx, tok);
    SODHIP_TRY_HIP(hipGetLastError());
    return SODHIP_OK;
}

extern "C" int sodhip_ducros_visc_limit_f64(sodhip_ctx ctx, int porder, int nelem, int npoin,
                                            const int *connec, const double *u,
                                            const double *divU, const double *vorti,
                                            const double *Ml, const double *helem,
                                            double ducros_min_val, double *mu_e)
{
    SODHIP_REQUIRE(ctx, "null context");
    SODHIP_REQUIRE(porder >= 2 && porder <= kMaxP, "porder %d not supported (2..4)", porder);
    SODHIP_REQUIRE(nelem > 0 && npoin > 0, "invalid mesh sizes");
    SODHIP_REQUIRE(connec && u && divU && vorti && Ml && helem && mu_e, "null array argument");
    SODHIP_TRY_HIP(hipSetDevice(ctx->device));
    MeshCache *m = nullptr;
    int rc = get_mesh(ctx, porder, nelem, npoin, connec, &m);
    if (rc) return rc;
    // the node pass's three arrays in the element-node scratch (3 npoin doubles,
    // far below the stage's records; the limiter runs between stages)
    if ((rc = ensure_buf(ctx->scratch, 3 * (size_t)npoin * sizeof(double)))) return rc;
    double *nq = (double *)ctx->scratch.ptr;
    int tok = prof_begin(ctx, 2);
    k_ducros_node<<<(npoin + 255) / 256, 256, 0, ctx->stream>>>(npoin, u, divU, vorti, Ml, nq);
#define SODHIP_DUCROS(KA, W) \
    k_ducros<KA, W><<<tile_grid(nelem, ctx->num_cu, W), 256, 0, ctx->stream>>>( \
        nelem, nnode_of(porder), porder, npoin, connec, m->perm, nq, helem, \
        ducros_min_val, mu_e)
    if (wide_tiles(nelem, ctx->num_cu)) SODHIP_BY_LINE(porder, SODHIP_DUCROS, kWideTile);
    else SODHIP_BY_LINE(porder, SODHIP_DUCROS, kTile);
#undef SODHIP_DUCROS
    prof_end(ctx, tok);
    SODHIP_TRY_HIP(hipGetLastError());
    return SODHIP_OK;
}
