// ops_element.hip -- element kernels of the split-form convection, the viscous
// operator and the generic scalar convection, the node-ordered assembly gather,
// and their drop-in C-ABI entry points.
//
// All operators, the fused stages at every order among them, run on the element
// pipeline of pipe.hpp (lane-per-node, line order, geometry through LDS): k_rhs the
// right-hand sides, k_grad the first-derivative operators; the opt-in brick-local
// assembly of the p=3 FP64 stage has a kernel of its own (k_rhs_split).  Element
// residuals go to a scratch array of 5-field records per element-node (whole elements:
// coalesced writes); a second kernel gathers them per node through the node-ordered
// incidence table in the reference's serial (element, node) order -- deterministic, no
// atomics.
//
// Arithmetic restatement: the split forms are evaluated through identities that
// hold for arbitrary nodal inputs (linearity of the discrete derivative and
// reordering of finite sums), which remove redundant work of the reference loop:
//  * the enthalpy-slot and kinetic-energy terms of the energy equation share one
//    derivative of H = E + k and of rho*H;
//  * advective derivatives a.grad(f) use contravariant components
//    sum_j He(j,k) a_j at the quadrature point;
//  * flux divergences sum_j d_j(s u_j) are evaluated from the line values of s
//    times the contravariant velocity sum_j He_g(j,k) u_j(m) at the line node m,
//    with the advective derivative of s folded into the same line sum (k_rhs).
#include <cstdio>
#include <type_traits>

#include "common.hpp"
#include "device.hpp"
#include "element.hpp"
#include "pipe.hpp"

namespace sodhip {

template <typename T> struct RhsArgs {
    int nelem, npoin;
    const int *connecT;
    const T *He, *gpvol, *dl;
    const int *inv, *gI, *gJ, *gK;
    // primitive inputs (drop-in operators)
    const T *u, *q, *rho, *pr, *E;
    const T *rho_n, *Tem, *mu_fluid, *mu_e, *mu_sgs;
    T Cp, Pr, c_rho, c_ener;
    // conserved inputs (fused stage): FP64 state
    const double *cr, *cq, *cE;
    double gamma, Rgas, mu_factor, p_ref;
    // per-element Sutherland factor (an ensemble of meshes whose instances
    // differ in it), or nullptr for the uniform mu_factor
    const double *mu_factor_e;
    const int *perm; // element-local scratch position of each node
    T *out;          // records of 5 (mass, mom1, mom2, mom3, energy) per element-node;
                     // (e,a) at record e*NN + perm[a]
    int run, wide;   // unit_range
    int geo16;       // He and gpvol blocks of every element are 16-byte aligned
    // brick-local assembly of the fused p=3 stage (see ClusterTables): the
    // element order, local-node tables, the partial records of surface nodes,
    // and the stage update the element kernel applies to interior nodes
    // (the arithmetic of k_gather_update)
    const int *cel, *cloc, *cnb, *cnode, *ckind;
    int ncl;
    double *rec;
    const double *invMl;
    double fact, lam1, lams, gdt;
    int rd1, rdy;
    const double *y1r, *y1q, *y1E;
    double *yr, *yq, *yE;
    double *Rm, *Rq, *Re;
    double nx_l1, nx_gdt;
    double *nxr, *nxq, *nxE;
    // LPS operators: node projection records (kProjRec values; the fused stage),
    // comp_tau's tau_stab, c_lps
    const double *prj, *tau;
    double c_lps;
    const double *pMass, *pEner, *pMX, *pMY, *pMZ; // or arrays (npoin,3) (drop-in)
};

// Sutherland's law (mod_fluid_viscosity.f90:21-41)
template <typename T> __device__ __forceinline__ T sutherland(T mu_factor, T Tk)
{
    return mu_factor * T(0.000001458) * (Tk * sqrt(Tk)) / (Tk + T(110.4));
}

// The operators of one right-hand side on the element pipeline (pipe.hpp).
// CONV: split-form convection (full_convec_ijk).  VISC: 1 the viscous operator
// (full_diffusion_ijk); 2 its LPS-stabilised form (full_diff_stab_ijk,
// elem_stab.f90:207-438); 3 full_proj_ijk's element part (elem_stab.f90:489-563),
// records of 12 values: gpvol times the upper triangle t11 t12 t13 t22 t23 t33 of
// 2 S - 2/3 div u I, grad rho and grad T.  CONS: inputs are the conserved FP64 state (the fused
// stage forms the primitives of updateF's EOS block and Sutherland's viscosity
// in-kernel) instead of the primitive arrays.
//
// Convection in two line coefficients.  With D_k(m) the derivative row of the
// lane's k-line, U_k = sum_j He(j,k) u_j(own), Q_k the same of q, and
// U_k(m) = sum_j He(j,k) u_j(m) at the line node m, the split form's terms
//   rho div(s u) + q.grad s   (s = u_i and H)     carry  E_k(m) = D_k(m) (Q_k + rho U_k(m)),
//   div(s u) + u.grad s       (s = q_i and rho H) carry  C_k(m) = D_k(m) (U_k + U_k(m)),
// so each of the eight fields costs one multiply-add per line node, and no
// line weight is kept: 22 multiply-adds per line node, where separate
// derivatives and W-weighted sums took 36 and held the weights in registers.
// The fused FP64 stage has q = rho u and rho H itself: with z = D_k(m) (U_k + U_k(m))
// the two coefficients meet in K = z (rho + rho(m)) on the four fields u_i and H,
// and div q + u.grad rho = sum z rho(m): 14 multiply-adds and seven values read per
// line node instead of 22 and eleven.
//
// Per unit, in phases (a workgroup of one wave has no barriers):
//   in      the unit's geometry (LDS), state (registers) and node ids (LDS) have
//           arrived; He and gpvol go to registers, the previous unit's residual
//           records leave LDS, and the copies and gathers of the next units start;
//   stage   nodal records -> LDS: u1 u2 | u3 rho | p H | rhoH q1 | q2 q3 (80 bytes
//           in FP64: 16 consecutive records start in 16 different banks);
//   lines   convection and the line derivatives of u, rho and T;
//   fluxes  G_k(F) = gpvol sum_d He(d,k) F_d -> LDS over the nodal records, the own
//           node's share of the weak divergence kept in registers;
//   weak    sum_k sum_b dl(b,k,I_k(a)) G_k(F)(b);
//   out     residual records -> LDS, dense, written by the next "in".
//
// What bounds it: the convection moves 8 GB between L1 and L2 at 553k elements, p=3
// (5 GB of them from HBM) and waits for them most of the time; it runs at about
// 5 TB/s of HBM traffic against 5.7 TB/s of a large copy.  The kernel of both
// operators adds LDS reads (51 of 16 bytes per lane at p=4) and FP64 arithmetic.  Against
// one element per workgroup in gmsh lane order with W-weighted sums, and geometry
// in 4-byte rows at odd p=4 elements (kernel times, one box):
//   p=3 FP64, 553k elements: convection 1.64 -> 1.14 ms, viscous 1.94 -> 1.28 ms
//   p=4 FP64,  63k elements: convection 0.77 -> 0.32 ms, viscous 0.80 -> 0.34 ms
//   p=4 FP32,  46k elements: convection 0.30 -> 0.15 ms, viscous 0.36 -> 0.18 ms
//   both, fused stage: p=4 FP64, 48k elements 1.57 -> 0.30 ms (it spilled 124
//   registers; 0.42 ms with q and rho H as fields of their own); p=2 FP64, 152k elements
//   0.47 -> 0.15 ms; p=3 FP64, 262k elements 0.83 -> 0.64 ms and p=3 with FP32
//   operators, 87k elements 0.21 -> 0.17 ms against two waves per element, one per
//   operator, that hand over through LDS.  The group's viscosities come together
//   (mu_issue): with every lane reading its own the p=3 kernels touched 64 lines per
//   element and array and took 0.76 ms (fused) and 1.54 ms (viscous).
//   LPS: p=4, 41k elements, convection and stabilised operator 0.77 (two kernels, the
//   second adding to the first one's records) -> 0.40 ms, projections 0.36 -> 0.20 ms;
//   p=3, 111k elements, 0.55 (two waves per element) -> 0.34 ms and 0.41 -> 0.27 ms;
//   drop-in stabilised operator p=4, 28k elements 0.38 -> 0.24 ms (these read He with
//   72-byte strides per lane).
template <int P, typename T, bool CONV, int VISC, bool CONS> struct ElemLDS {
    using Q = EP<P, T>;
    // nodal records (values), flux records and residual records share one area
    // of one stride, so that a line neighbour has one LDS offset
    // A group's units take their nodes together, line by line over the group's
    // elements (a gather's consecutive lanes then follow an i-line through G
    // neighbours and share its cache lines), where nothing but gathers and geometry is
    // read: the drop-in convection takes 1.14 instead of 1.25 ms (p=3, 553k elements)
    // and 321 instead of 336 us (p=4, 63k), the projections 266 instead of 269 us.  The
    // two barriers that this costs are not paid back in the kernels with a viscous flux:
    // 1.27 against 1.28 ms drop-in, and the fused stage 665 against 640 us (p=3, 262k)
    // and 312 against 300 us (p=4, 48k).  The areas of a group's units start 16 banks
    // apart.
    static constexpr bool JOINT = Q::G > 1 && (VISC == 0 || VISC == 3);
    static constexpr int REC = VISC == 3 ? 12 : VISC ? 18 : 10,
                         AREA = REC * Q::NT + (JOINT ? 64 / (int)sizeof(T) : 0);
    // at p=4 the transposed coefficients of both operators' kernel do not fit in
    // the registers beside the rest: they stay in LDS, one column per lane
    static constexpr bool TLDS = CONV && VISC && P == 4;
    // the fused LPS stage reads each node's projections as one 96-byte record
    // (kProjRec); they come through LDS in 16-byte pieces, consecutive lanes on
    // consecutive pieces, into the geometry's buffer once He is in registers (the
    // next geometry then follows them)
    static constexpr bool PJ = VISC == 2 && CONS;
    static constexpr int PROWS = (6 * Q::NL + 63) / 64, PI = (PROWS + Q::NW - 1) / Q::NW;
    static constexpr int GEO = PJ && PI * Q::NW * 1024 > Q::GEO ? PI * Q::NW * 1024 : Q::GEO;
};

// Values per residual record of the fused stage's element kernel.  With FP32
// operators at p=3 the five residuals are padded to six, so that a record starts on
// an 8-byte boundary and the stage's gather reads it with three 8-byte loads (the
// gather then takes 0.25 instead of 0.43 ms at 64^3 elements); in FP64 the 20 %
// larger records cost the element kernel more than the gather gains, and the
// drop-in operators' FP32 gather gains nothing (p=4, 46k elements: 51 us against
// 47 us with five).
template <int P, typename T> constexpr int stage_rw() { return sizeof(T) == 4 && P == 3 ? 6 : 5; }

// waves per SIMD asked of the compiler: the FP64 kernels hold He, the three
// derivative rows and the unit's state in registers
template <int P, typename T, bool CONV, int VISC> constexpr int elem_waves()
{
    return sizeof(T) == 4 || (VISC == 3 && !CONV) ? 3 : 2;
}

template <int P, typename T, bool CONV, int VISC, bool CONS>
__global__ __launch_bounds__((EP<P, T>::NTB), (elem_waves<P, T, CONV, VISC>())) void k_rhs(RhsArgs<T> A)
{
    using Q = EP<P, T>;
    using L = ElemLDS<P, T, CONV, VISC, CONS>;
    constexpr bool FLUX = VISC == 1 || VISC == 2, LPS = VISC == 2, PROJ = VISC == 3;
    static_assert(!(LPS || PROJ) || sizeof(T) == 8, "LPS: FP64");
    constexpr int GEO = L::GEO;
    using V2 = T __attribute__((ext_vector_type(2)));
    constexpr int NN = Q::NN, NL = Q::NL, NT = Q::NT, NE = Q::NE, NW = Q::NW, G = Q::G;
    constexpr int REC = L::REC, RW = PROJ ? 12 : CONS ? stage_rw<P, T>() : 5;
    // q = rho u and rho H formed from the other values, in FP64 only: in FP32 the
    // separately rounded q and u average their rounding errors (q of a 0.2-Mach flow
    // is 20 to 45 % less exact without)
    constexpr bool RHOU = CONS && sizeof(T) == 8;
    constexpr int TEM = 10; // temperature's place in the nodal record
    constexpr bool DELTA = sizeof(T) == 4; // differences to the own node's values
    // sums over the three lines, and products with the own node's values
    constexpr bool WIDE = DELTA && !CONS;
    using S = std::conditional_t<WIDE, double, T>;
    __shared__ __attribute__((aligned(16))) T area_s[G * L::AREA];
    __shared__ __attribute__((aligned(16))) unsigned char geo_s[G * GEO];
    __shared__ int conn_s[G * 2 * NT];
    // viscosities of the group's elements, [array][node][element]; by turns in two
    // places where no barrier separates their reads from the next copies
    constexpr bool MUS = FLUX && G > 1;
    constexpr int NMU = CONS ? 1 : 2, MUB = MUS ? (NN * G * (int)sizeof(T) + 255) / 256 * 256 : 0;
    constexpr int MUN = NW > 1 ? 1 : 2;
    __shared__ __attribute__((aligned(16))) unsigned char mu_s[MUS ? MUN * NMU * MUB : 4];
    // this thread's unit of the group, and its LDS
    const int sb = __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    T *const area = area_s + sb * L::AREA;
    unsigned char *const geo = geo_s + sb * GEO;
    int *const conn = conn_s + sb * 2 * NT;
    const unsigned geo_at = lds_addr(geo_s) + sb * GEO;
    const unsigned conn_at = lds_addr(conn_s) + sb * 2 * NT * 4;
    const int lane = threadIdx.x % NT, wl = lane & 63;
    const int wv = __builtin_amdgcn_readfirstlane(lane >> 6);

    const int nunits = (A.nelem + NE - 1) / NE;
    // over groups of G consecutive units; past the last unit it is evaluated
    // again, and not stored
    const UnitRange er = unit_range((nunits + G - 1) / G, A.run, A.wide);
    auto unit = [&](int g) { return min(g * G + sb, nunits - 1); };
    if (er.begin >= er.end) return;
    const int ulast = er.begin + (er.end - 1 - er.begin) / er.stride * er.stride;
    const LexLane<P, T, FLUX> ln(lane, A.dl, A.inv, A.perm);
    const size_t EN = (size_t)A.nelem * NN, np = (size_t)A.npoin;
    auto conn_issue = [&](int u, int slot) {
        const size_t i = (size_t)u * NL + lane;
        dma_lds<4>(A.connecT + (i < EN ? i : EN - 1), conn_at + (slot * NT + wv * 64) * 4);
    };
    // The element-fastest (nelem, nnode) viscosities of group g, G neighbours at a time:
    // the lanes of one row copy 256 bytes of [node][element], 4 each
    auto mu_issue = [&](int g, int slot) {
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
#pragma unroll
        for (int r0 = 0; r0 < MUB / 256; r0 += Q::NTB / 64) {
            const int r = r0 + wave, b = r * 256 + 4 * wl;
            if (MUB / 256 % (Q::NTB / 64) != 0 && r >= MUB / 256) break;
            const int node = min(b / (G * (int)sizeof(T)), NN - 1), in = b % (G * (int)sizeof(T));
            const size_t at = (size_t)min(g * G + in / (int)sizeof(T), A.nelem - 1) + (size_t)A.nelem * node;
            const unsigned to = lds_addr(mu_s) + slot % MUN * NMU * MUB + r * 256;
            dma_lds<4>((const char *)(A.mu_e + at) + in % (int)sizeof(T), to);
            if constexpr (!CONS)
                if (A.mu_sgs) dma_lds<4>((const char *)(A.mu_sgs + at) + in % (int)sizeof(T), to + MUB);
        }
    };
    __shared__ T tcol[L::TLDS ? 3 * P * Q::NT : 1];
    if constexpr (L::TLDS)
        if (sb == 0)
#pragma unroll
            for (int i = 0; i < 3 * P; ++i) tcol[i * NT + lane] = ln.t[i / P][i % P];
    int nb[3][P]; // LDS offsets of the line neighbours' records
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int o = 0; o < P; ++o) nb[k][o] = ln.nb[k][o] * REC;
    // the fused LPS stage: this lane's pieces of the unit's projection records, by the
    // place of their node in the unit's row of node ids
    __shared__ int pj_node[L::PJ ? L::PI * NT : 1];
    if constexpr (L::PJ)
        if (sb == 0)
            for (int i = 0; i < L::PI; ++i) {
                const int l = min(((wv + NW * i) * 64 + wl) / 6, NL - 1);
                pj_node[i * NT + lane] = l / NN * NN + min(max(A.inv[l % NN] - 1, 0), NN - 1);
            }
    auto ld2 = [&](int i) { return *(const V2 *)(area + i); };
    auto st2 = [&](int i, T x, T y) { *(V2 *)(area + i) = V2{x, y}; };

    // The node whose inputs this thread reads (one group of units ahead) and stages
    constexpr bool JOINT = L::JOINT;
    int gu = sb, gl = lane, ga = ln.a; // unit of the group, record, node
    if constexpr (JOINT) {
        constexpr int N1 = Q::N1, PAD = NT - NN;
        const int t = threadIdx.x, line = t / (G * N1), r = t % (G * N1);
        gu = r / N1;
        gl = line * N1 + r % N1;
        if (PAD > 0 && line >= N1 * N1) { // threads without a node fill the padding
            gu = (t - G * NN) / PAD;
            gl = NN + (t - G * NN) % PAD;
        }
        ga = min(max(A.inv[gl < NN ? gl : 0] - 1, 0), NN - 1);
    }
    T *const garea = area_s + gu * L::AREA + gl * REC;
    const int *const gconn = conn_s + gu * 2 * NT + (JOINT ? ga : ln.sub * NN + ln.a);
    struct In {
        double cr, cq[3], cE;                     // conserved state (CONS)
        T rho, u[3], q[3], pr, E, Tem, rhon, muf; // primitive inputs (drop-in)
        T mue, musgs;
        double tau; // LPS, own unit
        int n;      // own node
    };
    auto load = [&](In &x, int g, int slot) {
        const int n = gconn[slot * NT];
        if constexpr (CONS) {
            x.cr = A.cr[n];
            x.cq[0] = A.cq[n];
            x.cq[1] = A.cq[n + np];
            x.cq[2] = A.cq[n + 2 * np];
            x.cE = A.cE[n];
        } else {
            x.rho = A.rho[n];
#pragma unroll
            for (int d = 0; d < 3; ++d) x.u[d] = A.u[n + np * d];
            if constexpr (CONV) {
#pragma unroll
                for (int d = 0; d < 3; ++d) x.q[d] = A.q[n + np * d];
                x.pr = A.pr[n];
                x.E = A.E[n];
            }
            if constexpr (VISC != 0) x.Tem = A.Tem[n];
            if constexpr (FLUX) {
                x.rhon = A.rho_n[n];
                x.muf = A.mu_fluid[n];
            }
            if constexpr (LPS) x.n = conn[slot * NT + ln.sub * NN + ln.a];
        }
        const int e = min(unit(g) * NE + ln.sub, A.nelem - 1);
        if constexpr (LPS) x.tau = A.tau[e];
        if constexpr (FLUX && !MUS) {
            const size_t eg = (size_t)e + (size_t)A.nelem * ln.a;
            x.mue = A.mu_e[eg];
            if constexpr (!CONS) x.musgs = A.mu_sgs ? A.mu_sgs[eg] : T(0);
        }
    };
    using O = RecOut<P, T, RW>; // residual records

    In cur, nxt;
    GeoAt at = geo_issue<P, T>(A.He, A.gpvol, A.nelem, nunits, A.geo16, unit(er.begin), geo_at, wl, wv);
    conn_issue(unit(er.begin), 0);
    conn_issue(unit(min(er.begin + er.stride, ulast)), 1);
    if constexpr (MUS) mu_issue(er.begin, 0);
    wait_vm<0>();
    lds_barrier();
    load(cur, er.begin, 0);
    int slot = 1, prev = -1;
    for (int g = er.begin; g < er.end; g += er.stride, slot ^= 1) {
        const int u = unit(g), u2 = unit(min(g + er.stride, ulast)),
                  u3 = unit(min(g + 2 * er.stride, ulast));
        // ---------------- in
        wait_vm<0>();
        lds_barrier();
        T He[3][3];
        {
            const T *hp = (const T *)(geo + at.he) + 9 * (ln.sub * NN + ln.a);
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int i = 0; i < 3; ++i) He[i][j] = hp[i + 3 * j];
        }
        const T vol = ((const T *)(geo + Q::HEA + at.gv))[ln.sub * NN + ln.a];
        if constexpr (MUS) {
            const T *m = (const T *)(mu_s + (slot ^ 1) % MUN * NMU * MUB) + ln.a * G + sb;
            cur.mue = m[0];
            if constexpr (!CONS) cur.musgs = A.mu_sgs ? m[MUB / sizeof(T)] : T(0);
        }
        typename O::V out[O::NC];
        O::read(out, area, lane);
        lds_done();
        if (prev >= 0) O::store(out, area, A.out, prev, A.nelem, lane);
        load(nxt, min(g + er.stride, ulast), slot);
        int pn[L::PJ ? L::PI : 1];
        if constexpr (L::PJ) {
#pragma unroll
            for (int i = 0; i < L::PI; ++i) pn[i] = conn[(slot ^ 1) * NT + pj_node[i * NT + lane]];
        }
        unit_sync<JOINT ? 2 : NW>(); // (of a group: every unit's records have been read)
        if constexpr (MUS) mu_issue(min(g + er.stride, ulast), slot);
        if constexpr (L::PJ) {
#pragma unroll
            for (int i = 0; i < L::PI; ++i) {
                const int r = wv + NW * i;
                dma_lds<16>(A.prj + kProjRec * (size_t)pn[i] + 2 * ((r * 64 + wl) % 6), geo_at + r * 1024);
            }
        } else {
            at = geo_issue<P, T>(A.He, A.gpvol, A.nelem, nunits, A.geo16, u2, geo_at, wl, wv);
            conn_issue(u3, slot ^ 1);
        }
        // the drop-in LPS operator's projections, for the fluxes
        double pj[LPS ? 15 : 1]; // rows of the projected tensor, grad rho, grad T
        if constexpr (LPS && !CONS) {
            const double *pf[5] = {A.pMX, A.pMY, A.pMZ, A.pMass, A.pEner};
#pragma unroll
            for (int f = 0; f < 5; ++f)
#pragma unroll
                for (int d = 0; d < 3; ++d) pj[3 * f + d] = pf[f][cur.n + np * d];
        }
        prev = g * G + sb < nunits ? u : -1;
        // ---------------- stage
        T rho, v[3], q[3] = {0, 0, 0}, H = 0, rhoH = 0, p = 0, Tk = 0, muf = 0, rhon = 0, musgs = 0;
        const T mue = FLUX ? cur.mue : T(0);
        if constexpr (FLUX && !CONS) musgs = cur.musgs;
        if constexpr (CONS) {
            const double r = cur.cr, ri = 1.0 / r;
            double ud[3], umag = 0.0;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                ud[d] = cur.cq[d] * ri;
                umag += ud[d] * ud[d];
            }
            const double eint = cur.cE * ri - 0.5 * umag;
            const double pd = r * (A.gamma - 1.0) * eint;
            const double hd = (A.gamma / (A.gamma - 1.0)) * pd * ri;
            const double Td = pd * ri / A.Rgas;
            rho = T(r);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                v[d] = T(ud[d]);
                q[d] = T(cur.cq[d]);
            }
            // only grad p enters: a uniform reference pressure is removed
            // before the (possibly FP32) operator arithmetic
            p = T(pd - A.p_ref);
            H = T(hd + 0.5 * umag);
            rhoH = T(r * (hd + 0.5 * umag));
            Tk = T(Td);
            rhon = rho;
            muf = T(sutherland<double>(
                A.mu_factor_e ? A.mu_factor_e[min(u * NE + ln.sub, A.nelem - 1)] : A.mu_factor, Td));
        } else {
            rho = cur.rho;
#pragma unroll
            for (int d = 0; d < 3; ++d) v[d] = cur.u[d];
            if constexpr (CONV) {
#pragma unroll
                for (int d = 0; d < 3; ++d) q[d] = cur.q[d];
                p = cur.pr;
                H = cur.E + (v[0] * v[0] * T(0.5) + v[1] * v[1] * T(0.5) + v[2] * v[2] * T(0.5));
                rhoH = rho * H;
            }
            if constexpr (VISC != 0) Tk = cur.Tem;
            if constexpr (FLUX) {
                rhon = cur.rhon;
                muf = cur.muf;
            }
        }
        // (lanes without a node write records of their own past the unit's: a
        // condition here would let the compiler sink the arithmetic behind it)
        const int own = lane * REC;
        auto put = [&](int i, T x, T y) { *(V2 *)(garea + i) = V2{x, y}; };
        put(0, v[0], v[1]);
        put(2, v[2], rho);
        if constexpr (CONV) put(4, p, H);
        if constexpr (CONV && !RHOU) {
            put(6, rhoH, q[0]);
            put(8, q[1], q[2]);
        }
        if constexpr (VISC != 0) garea[TEM] = Tk;
        unit_sync<JOINT ? 2 : NW>();
        if constexpr (JOINT) { // back to the lane's own node
            const V2 x01 = ld2(own), x2r = ld2(own + 2);
            v[0] = x01.x;
            v[1] = x01.y;
            v[2] = x2r.x;
            rho = x2r.y;
            if constexpr (CONV) {
                const V2 xpH = ld2(own + 4);
                p = xpH.x;
                H = xpH.y;
            }
            if constexpr (CONV && !RHOU) {
                const V2 xHq = ld2(own + 6), xqq = ld2(own + 8);
                rhoH = xHq.x;
                q[0] = xHq.y;
                q[1] = xqq.x;
                q[2] = xqq.y;
            }
            if constexpr (VISC != 0) Tk = area[own + TEM];
        }

        // ---------------- lines
        T Rm = 0, Rq[3] = {0, 0, 0}, Re = 0;
        T du[3][3], dT[3]; // d u_i / d xi_k, d T / d xi_k
        T gR[3];           // grad rho
        {
            T Ut[3] = {0, 0, 0}, Qt[3] = {0, 0, 0}, dr[3], dp[3];
            // RHOU: divQ holds sum z rho(m) = div q + u.grad rho
            S divU = 0, divQ = 0;
            // Sums start with the own node's share.  FP32 sums the differences to the
            // own node's values (whose share is then the row sum rs of D, zero but for
            // rounding), so that a field's mean costs no digits of its derivative.
            // FP64 has digits to spare and sums the values.  On nodal noise, which has no
            // mean to remove, the differences' own rounding made the drop-in operators
            // less exact than separate derivatives are (error over result, p = 2, 3, 4:
            // convection's energy 7.2e-8 -> 8.5 to 8.8e-8, viscous momentum 5.9, 6.6,
            // 7.1e-8 -> 6.6, 7.6, 8.4e-8); with the sums over the lines and the closing
            // products in FP64 (S, WIDE) they are 6.9 to 7.1e-8 and 5.8, 6.4, 6.9e-8
            // (46k elements, p=4, both operators: 402 -> 405 us; 2.1M, convection: 8.5 ->
            // 8.7 ms).
            // The fused stage, whose states are smooth, is more exact than with separate
            // derivatives as it is (a step's state by 10 to 30 %), and FP64 sums cost it
            // 2 % of its time (87k elements, p=3: 1.72 -> 1.76 ms per step).
            T rs[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                double r = ln.ds[k]; // in 64 bits: the coefficients all but cancel
                if constexpr (DELTA)
#pragma unroll
                    for (int o = 0; o < P; ++o) r += ln.d[k][o];
                rs[k] = T(r);
            }
            T a0 = 0, b0 = 0;
            if constexpr (CONV) {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    Ut[k] = He[0][k] * v[0] + He[1][k] * v[1] + He[2][k] * v[2];
                    if constexpr (!RHOU) Qt[k] = He[0][k] * q[0] + He[1][k] * q[1] + He[2][k] * q[2];
                    a0 += rs[k] * Ut[k];
                    b0 += rs[k] * Qt[k];
                }
                divU = a0;
                divQ = RHOU ? T(2) * rho * a0 : b0;
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                // sums of one line first: shorter chains of roundings
                T rq[3] = {0, 0, 0}, re = 0, dvu = 0, dvq = 0;
                // E = c (eb + rho u'), C = c (cb + u') with u' = U_k(m), or its
                // difference to U_k
                const T eb = DELTA ? Qt[k] + rho * Ut[k] : Qt[k], cb = DELTA ? T(2) * Ut[k] : Ut[k];
                dr[k] = rs[k] * rho;
                if constexpr (CONV) dp[k] = rs[k] * p;
                if constexpr (VISC != 0) {
                    dT[k] = rs[k] * Tk;
#pragma unroll
                    for (int i = 0; i < 3; ++i) du[i][k] = rs[k] * v[i];
                }
#pragma unroll
                for (int o = 0; o < P; ++o) {
                    const int b = nb[k][o];
                    const T c = ln.d[k][o];
                    V2 x01 = ld2(b), x2r = ld2(b + 2);
                    if constexpr (DELTA) {
                        x01 -= V2{v[0], v[1]};
                        x2r -= V2{v[2], rho};
                    }
                    dr[k] += c * x2r.y;
                    if constexpr (CONV && RHOU) {
                        const V2 xpH = ld2(b + 4);
                        const T ut = He[0][k] * x01.x + He[1][k] * x01.y + He[2][k] * x2r.x;
                        const T z = c * (Ut[k] + ut), K = z * (rho + x2r.y);
                        dvu += c * ut;
                        dvq += z * x2r.y;
                        rq[0] += K * x01.x;
                        rq[1] += K * x01.y;
                        rq[2] += K * x2r.x;
                        re += K * xpH.y;
                        dp[k] += c * xpH.x;
                    } else if constexpr (CONV) {
                        V2 xpH = ld2(b + 4), xHq = ld2(b + 6), xqq = ld2(b + 8);
                        if constexpr (DELTA) {
                            xpH -= V2{p, H};
                            xHq -= V2{rhoH, q[0]};
                            xqq -= V2{q[1], q[2]};
                        }
                        const T ut = He[0][k] * x01.x + He[1][k] * x01.y + He[2][k] * x2r.x;
                        const T qt = He[0][k] * xHq.y + He[1][k] * xqq.x + He[2][k] * xqq.y;
                        dvu += c * ut;
                        dvq += c * qt;
                        const T C = c * (cb + ut), E = c * (eb + rho * ut);
                        rq[0] += E * x01.x;
                        rq[1] += E * x01.y;
                        rq[2] += E * x2r.x;
                        re += E * xpH.y;
                        re += C * xHq.x;
                        rq[0] += C * xHq.y;
                        rq[1] += C * xqq.x;
                        rq[2] += C * xqq.y;
                        dp[k] += c * xpH.x;
                    }
                    if constexpr (VISC != 0) {
                        du[0][k] += c * x01.x;
                        du[1][k] += c * x01.y;
                        du[2][k] += c * x2r.x;
                        dT[k] += c * (DELTA ? area[b + TEM] - Tk : area[b + TEM]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (CONV) {
#pragma unroll
                    for (int i = 0; i < 3; ++i) Rq[i] += rq[i];
                    Re += re;
                    divU += dvu;
                    divQ += dvq;
                }
            }
            if constexpr (VISC != 0)
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    gR[i] = He[i][0] * dr[0] + He[i][1] * dr[1] + He[i][2] * dr[2];
            if constexpr (CONV && RHOU) {
                // the own values' coefficient: s + rho div u and the own share of sum K
                const T s = divQ, B = s + rho * (divU + T(4) * a0);
                Rm = vol * (T(0.5) * (s + rho * divU));
                Re = vol * (T(0.25) * (Re + H * B));
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    Rq[i] = vol * (T(0.25) * (Rq[i] + v[i] * B) +
                                   (He[i][0] * dp[0] + He[i][1] * dp[1] + He[i][2] * dp[2]));
            } else if constexpr (CONV) {
                const S urho = S(Ut[0]) * dr[0] + S(Ut[1]) * dr[1] + S(Ut[2]) * dr[2];
                const S s = divQ + urho;
                // the own values' coefficients: div q + u.grad rho for u_i and H,
                // div u for q_i and rho H, and the own share of sum E and sum C (all of
                // it where differences are summed)
                const S ce = s + (b0 + rho * (DELTA ? divU : a0));
                const S cc = DELTA ? S(2) * divU + a0 : divU + S(2) * a0;
                Rm = T(vol * (S(0.5) * (s + rho * divU)));
                Re = T(vol * (S(0.25) * (Re + (H * ce + rhoH * cc))));
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    Rq[i] = T(vol * (S(0.25) * (Rq[i] + (v[i] * ce + q[i] * cc)) +
                                     (He[i][0] * dp[0] + He[i][1] * dp[1] + He[i][2] * dp[2])));
            }
        }

        if constexpr (CONV && LPS) {
            // formed here, not where they are used: sunk past the copies' branches
            // below they would keep the convection's inputs alive
            pin(Rm);
            pin(Re);
#pragma unroll
            for (int i = 0; i < 3; ++i) pin(Rq[i]);
        }
        double po[PROJ ? 12 : 1];
        if constexpr (VISC != 0) {
            // physical gradients: gU[i][j] = d u_i / d x_j, and grad T
            T gU[3][3], gt[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
#pragma unroll
                for (int j = 0; j < 3; ++j)
                    gU[i][j] = He[j][0] * du[i][0] + He[j][1] * du[i][1] + He[j][2] * du[i][2];
                gt[i] = He[i][0] * dT[0] + He[i][1] * dT[1] + He[i][2] * dT[2];
            }
            const T dv = gU[0][0] + gU[1][1] + gU[2][2];
            if constexpr (PROJ) {
                int f = 0;
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int d = i; d < 3; ++d)
                        po[f++] = vol * (gU[i][d] + gU[d][i] - (i == d ? (2.0 / 3.0) * dv : 0.0));
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    po[6 + d] = vol * gR[d];
                    po[9 + d] = vol * gt[d];
                }
            }
            if constexpr (FLUX) {
            // ---------------- fluxes.  Record per k: grad rho, grad T | tau u, tau_1 |
            // tau_2, tau_3 (contravariant, times gpvol)
            T W[6] = {0, 0, 0, 0, 0, 0};
            const T mufg = muf + rhon * musgs, mut = mufg + mue;
            const T kappa = muf * A.Cp / A.Pr + A.c_ener * mue * A.Cp / A.Pr +
                            A.Cp * rhon * musgs / T(0.9);
            if constexpr (L::PJ) wait_vm<0>(); // the projections
            if constexpr (NW > 1) lds_barrier(); // every wave has read the nodal records
            if constexpr (LPS) {
                // per point (nu_e and kappa_e inside): the stabilising terms -c_lps tau
                // (Proj - grad), times rho for momentum and rho Cp/Pr for energy.
                // Record per k: mass, energy | momentum 1, 2 | 3
                const T cl = -A.c_lps * cur.tau, clr = cl * rhon, tt = T(2.0 / 3.0) * dv;
                const T nu_e = A.c_rho * mue / rhon, cle = clr * A.Cp / A.Pr;
                // projection j of the node (rows of the tensor from its upper triangle)
                auto prj = [&](int j) -> T {
                    if constexpr (L::PJ) {
                        const int tri[15] = {0, 1, 2, 1, 3, 4, 2, 4, 5, 6, 7, 8, 9, 10, 11};
                        return ((const T *)(geo + 96 * lane))[tri[j]];
                    } else {
                        return pj[j];
                    }
                };
                T h[3][3], tu[3] = {0, 0, 0};
#pragma unroll
                for (int k = 0; k < 3; ++k)
#pragma unroll
                    for (int d = 0; d < 3; ++d) h[k][d] = vol * He[d][k];
                // flux f (its three components F) to the records and its own share of W;
                // one flux at a time, to keep few values alive
                auto flux = [&](int f, int at, const T F[3]) {
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        const T X = h[k][0] * F[0] + h[k][1] * F[1] + h[k][2] * F[2];
                        W[f] += ln.ds[k] * X;
                        area[own + 6 * k + at] = X;
                    }
                    __builtin_amdgcn_sched_barrier(0);
                };
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    T F[3];
#pragma unroll
                    for (int d = 0; d < 3; ++d) {
                        const T S = gU[i][d] + gU[d][i], St = i == d ? S - tt : S;
                        const T ts = i == d ? mut * S - mufg * tt : mut * S;
                        F[d] = clr * (prj(3 * i + d) - St) + ts;
                        tu[d] += ts * v[i];
                    }
                    flux(1 + i, 2 + i, F);
                }
                {
                    T F[3];
#pragma unroll
                    for (int d = 0; d < 3; ++d) F[d] = cl * (prj(9 + d) - gR[d]) + nu_e * gR[d];
                    flux(0, 0, F);
#pragma unroll
                    for (int d = 0; d < 3; ++d) F[d] = cle * (prj(12 + d) - gt[d]) + kappa * gt[d] + tu[d];
                    flux(4, 1, F);
                }
            } else {
                const T tt = mufg * T(2.0 / 3.0) * dv;
                T tau[3][3];
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 3; ++j) tau[i][j] = mut * (gU[i][j] + gU[j][i]);
#pragma unroll
                for (int i = 0; i < 3; ++i) tau[i][i] -= tt;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const T h0 = vol * He[0][k], h1 = vol * He[1][k], h2 = vol * He[2][k];
                    T F[6];
                    F[2] = 0;
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        F[3 + r] = h0 * tau[r][0] + h1 * tau[r][1] + h2 * tau[r][2];
                        F[2] += F[3 + r] * v[r]; // tau is symmetric: contravariant (tau u)_k
                    }
                    F[0] = h0 * gR[0] + h1 * gR[1] + h2 * gR[2];
                    F[1] = h0 * gt[0] + h1 * gt[1] + h2 * gt[2];
#pragma unroll
                    for (int f = 0; f < 6; ++f) W[f] += ln.ds[k] * F[f];
                    st2(own + 6 * k, F[0], F[1]);
                    st2(own + 6 * k + 2, F[2], F[3]);
                    st2(own + 6 * k + 4, F[4], F[5]);
                }
            }
            unit_sync<NW>();
            if constexpr (L::PJ) {
#pragma unroll
                for (int f = 0; f < 5; ++f) pin(W[f]);
                lds_done(); // this wave has read its projections; with a barrier, all have
                at = geo_issue<P, T>(A.He, A.gpvol, A.nelem, nunits, A.geo16, u2, geo_at, wl, wv);
                conn_issue(u3, slot ^ 1);
            }
            // ---------------- weak divergence
            S Ws[6]; // WIDE: the own share and the three lines' sums
            if constexpr (WIDE)
#pragma unroll
                for (int f = 0; f < 6; ++f) Ws[f] = W[f];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                T l[6] = {0, 0, 0, 0, 0, 0};
                T(&X)[6] = WIDE ? l : W;
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int o = 0; o < P; ++o) {
                    const int b = nb[k][o] + 6 * k;
                    const T c = L::TLDS ? tcol[(k * P + o) * NT + lane] : ln.t[k][o];
                    const V2 x01 = ld2(b), x23 = ld2(b + 2);
                    if constexpr (LPS) { // mass, momentum 1, 2, 3, energy
                        X[0] += c * x01.x;
                        X[4] += c * x01.y;
                        X[1] += c * x23.x;
                        X[2] += c * x23.y;
                        X[3] += c * area[b + 4];
                    } else {
                        const V2 x45 = ld2(b + 4);
                        X[0] += c * x01.x;
                        X[1] += c * x01.y;
                        X[2] += c * x23.x;
                        X[3] += c * x23.y;
                        X[4] += c * x45.x;
                        X[5] += c * x45.y;
                    }
                }
                if constexpr (WIDE)
#pragma unroll
                    for (int f = 0; f < 6; ++f) Ws[f] += l[f];
            }
            if constexpr (WIDE)
#pragma unroll
                for (int f = 0; f < 6; ++f) W[f] = T(Ws[f]);
            if constexpr (LPS) {
                Rm += W[0];
                Re += W[4];
#pragma unroll
                for (int i = 0; i < 3; ++i) Rq[i] += W[1 + i];
            } else {
                Rm += A.c_rho * mue / rhon * W[0];
                Re += W[2] + kappa * W[1];
#pragma unroll
                for (int i = 0; i < 3; ++i) Rq[i] += W[3 + i];
            }
            } // FLUX
        }
        // ---------------- out
        unit_sync<NW>(); // every wave is done with the records in `area`
        if constexpr (PROJ) {
#pragma unroll
            for (int i = 0; i < 6; ++i) st2(12 * ln.rec + 2 * i, po[2 * i], po[2 * i + 1]);
        } else {
            T *o = area + RW * ln.rec;
            if constexpr (RW == 6) o[5] = T(0);
            o[0] = Rm;
            o[1] = Rq[0];
            o[2] = Rq[1];
            o[3] = Rq[2];
            o[4] = Re;
        }
        cur = nxt;
    }
    lds_barrier();
    typename O::V out[O::NC];
    O::read(out, area, lane);
    if (prev >= 0) O::store(out, area, A.out, prev, A.nelem, lane);
    // no copy may still be writing this block's LDS when it retires
    wait_vm<0>();
}

// The first-derivative operators on the element pipeline, by OP:
//   SFUSED, SFLUX  generic_scalar_convec_ijk (elem_convec.f90:472-594):
//     gpvol [ 1/2 (div f + eta div u) + 1/2 u.grad(eta) ], with f = u eta formed in
//     registers (the time loop's f_eta = u(:,:,1) * eta(:,1) of the same two arrays)
//     or read;
//   DIV, CURL, DIVCURL  eval_divergence (mod_operators.f90:485-570) and
//     compute_vorticity (mod_operators.f90:684-775) at each GLL point.  With g_ik =
//     du_i/dxi_k the line derivatives and grad u(i,j) = sum_k He(j,k) g_ik: gpvol *
//     div u, and eps_ijk du_j/dx_k (the reference's leviCivi sum, minus the curl).
// Records of RW values per element-node at e*NN + perm[a].
//
// What bounds it: memory.  The 80 bytes of geometry per element-node are most of
// what is read; copied through LDS they are read once and in order, where each lane
// read its own 72 bytes of He at a stride of 72: entropy convection 432 -> 356 us
// (262k elements, p=3; 335 us at a large copy's rate), 250 -> 145 us (48k, p=4) and
// 143 -> 102 us (152k, p=2); DIVCURL 220 -> 127 us (41k, p=4).  CURL does not copy the
// gpvol that it does not read: the call 614 -> 591 us (262k, p=3), 410 -> 400 us (85k, p=4).
enum class GradOp { SFUSED, SFLUX, DIV, CURL, DIVCURL };

// waves per SIMD asked of the compiler: as many as run without spilling
template <int P, typename T, GradOp OP> constexpr int grad_waves()
{
    return sizeof(T) == 8 && (P == 4 || OP == GradOp::SFLUX) ? 3 : 4;
}

template <int P, typename T, GradOp OP>
__global__ __launch_bounds__((EP<P, T>::NTB), (grad_waves<P, T, OP>())) void k_grad(RhsArgs<T> A, const T *__restrict__ f,
                                                            const T *__restrict__ eta)
{
    using Q = EP<P, T>;
    using V2 = T __attribute__((ext_vector_type(2)));
    constexpr bool SC = OP == GradOp::SFUSED || OP == GradOp::SFLUX, FLUX = OP == GradOp::SFLUX;
    constexpr bool DIV = OP == GradOp::DIV || OP == GradOp::DIVCURL,
                   CURL = OP == GradOp::CURL || OP == GradOp::DIVCURL;
    constexpr int NN = Q::NN, NL = Q::NL, NT = Q::NT, NE = Q::NE, NW = Q::NW, G = Q::G;
    constexpr int RW = SC ? 1 : (DIV ? 1 : 0) + (CURL ? 3 : 0);
    constexpr bool VOL = SC || DIV; // the vorticity alone is not weighted
    // nodal records u1 u2 | u3 eta | f1 f2 | f3 -, at a stride of an odd number of
    // pairs, so that 16 consecutive records start in 16 different banks
    constexpr int REC = FLUX ? 10 : 6;
    __shared__ __attribute__((aligned(16))) T area_s[G * REC * NT];
    __shared__ __attribute__((aligned(16))) unsigned char geo_s[G * Q::GEO];
    __shared__ int conn_s[G * 2 * NT];
    const int sb = __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    T *const area = area_s + sb * REC * NT;
    unsigned char *const geo = geo_s + sb * Q::GEO;
    int *const conn = conn_s + sb * 2 * NT;
    const unsigned geo_at = lds_addr(geo_s) + sb * Q::GEO;
    const unsigned conn_at = lds_addr(conn_s) + sb * 2 * NT * 4;
    const int lane = threadIdx.x % NT, wl = lane & 63;
    const int wv = __builtin_amdgcn_readfirstlane(lane >> 6);

    const int nunits = (A.nelem + NE - 1) / NE;
    const UnitRange er = unit_range((nunits + G - 1) / G, A.run, A.wide);
    auto unit = [&](int g) { return min(g * G + sb, nunits - 1); };
    if (er.begin >= er.end) return;
    const int ulast = er.begin + (er.end - 1 - er.begin) / er.stride * er.stride;
    const LexLane<P, T, false> ln(lane, A.dl, A.inv, A.perm);
    const size_t EN = (size_t)A.nelem * NN, np = (size_t)A.npoin;
    auto conn_issue = [&](int u, int slot) {
        const size_t i = (size_t)u * NL + lane;
        dma_lds<4>(A.connecT + (i < EN ? i : EN - 1), conn_at + (slot * NT + wv * 64) * 4);
    };
    struct In {
        T et, u[3], fv[3];
    };
    auto load = [&](In &x, int slot) {
        const int n = conn[slot * NT + ln.sub * NN + ln.a];
        if constexpr (SC) x.et = eta[n];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            x.u[d] = A.u[n + np * d];
            if constexpr (FLUX) x.fv[d] = f[n + np * d];
        }
    };
    using O = RecOut<P, T, RW>;

    In cur, nxt;
    GeoAt at = geo_issue<P, T, VOL>(A.He, A.gpvol, A.nelem, nunits, A.geo16, unit(er.begin), geo_at, wl, wv);
    conn_issue(unit(er.begin), 0);
    conn_issue(unit(min(er.begin + er.stride, ulast)), 1);
    wait_vm<0>();
    lds_barrier();
    load(cur, 0);
    int slot = 1, prev = -1;
    for (int g = er.begin; g < er.end; g += er.stride, slot ^= 1) {
        const int u = unit(g), u2 = unit(min(g + er.stride, ulast)),
                  u3 = unit(min(g + 2 * er.stride, ulast));
        wait_vm<0>();
        lds_barrier();
        T He[3][3];
        {
            const T *hp = (const T *)(geo + at.he) + 9 * (ln.sub * NN + ln.a);
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int i = 0; i < 3; ++i) He[i][j] = hp[i + 3 * j];
        }
        const T vol = VOL ? ((const T *)(geo + Q::HEA + at.gv))[ln.sub * NN + ln.a] : T(1);
        typename O::V out[O::NC];
        O::read(out, area, lane);
        lds_done();
        if (prev >= 0) O::store(out, area, A.out, prev, A.nelem, lane);
        load(nxt, slot);
        unit_sync<NW>();
        at = geo_issue<P, T, VOL>(A.He, A.gpvol, A.nelem, nunits, A.geo16, u2, geo_at, wl, wv);
        conn_issue(u3, slot ^ 1);
        prev = g * G + sb < nunits ? u : -1;

        const T *v = cur.u;
        T fo[3] = {0, 0, 0};
        if constexpr (SC)
#pragma unroll
            for (int d = 0; d < 3; ++d) fo[d] = FLUX ? cur.fv[d] : v[d] * cur.et;
        const int own = lane * REC;
        *(V2 *)(area + own) = V2{v[0], v[1]};
        *(V2 *)(area + own + 2) = V2{v[2], SC ? cur.et : T(0)};
        if constexpr (FLUX) {
            *(V2 *)(area + own + 4) = V2{fo[0], fo[1]};
            area[own + 6] = fo[2];
        }
        unit_sync<NW>();

        // multiply-adds by name: SFUSED and SFLUX give the same bits whichever of two
        // products the compiler would contract
        T gE[3] = {0, 0, 0}, divU = 0, divF = 0, gu[3][3] = {}; // gu[i][j] = du_i/dx_j
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const T c0 = ln.ds[k];
            T de = SC ? c0 * cur.et : T(0), du[3], df[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                du[d] = c0 * v[d];
                df[d] = c0 * fo[d];
            }
#pragma unroll
            for (int o = 0; o < P; ++o) {
                const T *b = area + ln.nb[k][o] * REC;
                const T c = ln.d[k][o];
                const V2 x01 = *(const V2 *)b, x2e = *(const V2 *)(b + 2);
                const T x[3] = {x01.x, x01.y, x2e.x};
#pragma unroll
                for (int d = 0; d < 3; ++d) du[d] = fma(c, x[d], du[d]);
                if constexpr (SC) {
                    de = fma(c, x2e.y, de);
                    T y[3];
                    if constexpr (FLUX) {
                        const V2 f01 = *(const V2 *)(b + 4);
                        y[0] = f01.x;
                        y[1] = f01.y;
                        y[2] = b[6];
                    } else {
#pragma unroll
                        for (int d = 0; d < 3; ++d) y[d] = x[d] * x2e.y;
                    }
#pragma unroll
                    for (int d = 0; d < 3; ++d) df[d] = fma(c, y[d], df[d]);
                }
            }
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                if constexpr (SC) {
                    gE[i] = fma(He[i][k], de, gE[i]);
                    divU = fma(He[i][k], du[i], divU);
                    divF = fma(He[i][k], df[i], divF);
                } else {
#pragma unroll
                    for (int j = 0; j < 3; ++j) gu[i][j] += He[j][k] * du[i];
                }
            }
        }
        T r[RW];
        if constexpr (SC) {
            T t = T(0.5) * fma(cur.et, divU, divF);
#pragma unroll
            for (int i = 0; i < 3; ++i) t = fma(T(0.5), v[i] * gE[i], t);
            r[0] = vol * t;
        } else {
            int n = 0;
            if constexpr (DIV) r[n++] = vol * (gu[0][0] + gu[1][1] + gu[2][2]);
            if constexpr (CURL) {
                r[n++] = gu[1][2] - gu[2][1];
                r[n++] = gu[2][0] - gu[0][2];
                r[n++] = gu[0][1] - gu[1][0];
            }
        }
#pragma unroll
        for (int i = 0; i < RW; ++i) pin(r[i]);
        unit_sync<NW>();
#pragma unroll
        for (int i = 0; i < RW; ++i) area[ln.rec * RW + i] = r[i];
        cur = nxt;
    }
    lds_barrier();
    typename O::V out[O::NC];
    O::read(out, area, lane);
    if (prev >= 0) O::store(out, area, A.out, prev, A.nelem, lane);
    // no copy may still be writing this block's LDS when it retires
    wait_vm<0>();
}

// curlU(n,:) /= lelpn(n) over the working nodes (compute_vorticity's makeConti)
template <typename T>
__global__ __launch_bounds__(256) void k_per_elem_count(int npoin, int npoin_w,
                                                        const int *__restrict__ lpoin_w,
                                                        const int *__restrict__ lelpn,
                                                        T *__restrict__ curl)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npoin_w) return;
    const int n = lpoin_w[i] - 1;
    const T c = T(lelpn[n]);
#pragma unroll
    for (int d = 0; d < 3; ++d) curl[n + (size_t)npoin * d] /= c;
}

// Node-ordered assembly: R_f(n) = (init ? 0 : R_f(n)) + sum_j fact * scr[src[j]*NF + f], j
// over the node's slots row[n]..row[n+1]-1 in ascending (element, node) order
// (records of NF fields per element-node).  Slots are taken four at a time
// with every record load issued before the additions, which stay in slot
// order; blocks are mapped XCD-aware (the nodes of one XCD are one contiguous
// range, whose records share that XCD's L2).
template <typename TS, typename TR, int NF>
__global__ __launch_bounds__(256) void k_gather(int npoin, const int *__restrict__ row,
                                                const int *__restrict__ src,
                                                const TS *__restrict__ scr, TR *__restrict__ R0,
                                                TR *__restrict__ R1, TR *__restrict__ R2,
                                                TR *__restrict__ R3, TR *__restrict__ R4, int init,
                                                TR fact)
{
    const int per = gridDim.x >> 3; // grid is a multiple of 8
    const int blk = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    const int n = blk * blockDim.x + threadIdx.x;
    if (n >= npoin) return;
    const int j0 = row[n], j1 = row[n + 1];
    TR *R[5] = {R0, R1, R2, R3, R4};
    TR acc[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] = init ? TR(0) : R[f][n];
    for (int j = j0; j < j1; j += 4) {
        int sj[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) sj[u] = j + u < j1 ? src[j + u] : -1;
        TR v[4][NF];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if constexpr (NF == 5 && sizeof(TS) == 8) {
                // an absent slot reads record 0 (always present) and is not added
                double w[5];
                load_rec5((const double *)scr, max(sj[u], 0), w);
#pragma unroll
                for (int f = 0; f < NF; ++f) v[u][f] = TR(w[f]);
            } else {
                // an absent slot reads record 0 unconditionally (cheaper than
                // masking each load) and is not added
#pragma unroll
                for (int f = 0; f < NF; ++f) v[u][f] = TR(scr[(size_t)max(sj[u], 0) * NF + f]);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (sj[u] >= 0) {
#pragma unroll
                for (int f = 0; f < NF; ++f) acc[f] += fact * v[u][f];
            }
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) R[f][n] = acc[f];
}

// Tail of the entropy residual on the scalar gather (working nodes): the
// slots of node n summed as k_gather sums them, times invMl (lumped_solver_scal),
// then the residual of k_entropy_residual; Reta and eta are (npoin,2)
struct EntropyTail {
    int npoin_w;
    const int *lpoin_w;
    const double *invMl, *eta;
    double factor_comp, dt;
    double *Reta, *auxReta;
};

__global__ __launch_bounds__(256) void k_gather_entropy(int npoin, const int *__restrict__ wrow,
                                                        const int *__restrict__ wsrc,
                                                        const double *__restrict__ scr,
                                                        EntropyTail t, double fact)
{
    const int per = gridDim.x >> 3; // grid is a multiple of 8
    const int blk = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    const int i = blk * blockDim.x + threadIdx.x;
    if (i >= t.npoin_w) return;
    const int n = t.lpoin_w[i] - 1;
    const int j0 = wrow[i], j1 = wrow[i + 1];
    double acc = 0.0;
    for (int j = j0; j < j1; j += 4) {
        int sj[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) sj[u] = j + u < j1 ? wsrc[j + u] : -1;
        double v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = scr[max(sj[u], 0)]; // absent: record 0, not added
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (sj[u] >= 0) acc += fact * v[u];
    }
    const double r2 = acc * t.invMl[n];
    const double r1 = t.Reta[n];
    t.Reta[n + (size_t)npoin] = r2;
    t.auxReta[n] = (1.5 * r2 - 0.5 * r1) +
                   t.factor_comp * (t.eta[n + (size_t)npoin] - t.eta[n]) / t.dt;
    t.Reta[n] = r2;
}

// ---------------------------------------------------------------- launch helpers
// ---------------------------------------------------------------------------
// Element kernel of the brick-local assembly (the opt-in mode of the fused FP64
// stage at p=3).  Two waves share an element and its LDS: wave 0 evaluates the
// split-form convection, wave 1 the viscous operator and hands its residuals to wave 0
// through LDS; wave 0 puts their sum back as the element's records, and wave 1 adds
// those to the cluster's accumulator during the next element.  Each wave holds its own
// operator's live state, which leaves registers (214 of 256) for what the ring's copies
// and the accumulator's tables need.  Requires (p+1)^3 == 64: one wave per operator, one
// lane per node.
//
// The inputs stream through an LDS ring AH elements deep.  Every input of
// element e (He and gpvol, the five conserved fields at its nodes, mu_e) is
// copied global -> LDS by direct-to-LDS loads, which hold no registers while
// in flight, AH elements before e is evaluated; its connectivity row arrives
// AH elements earlier still, since the field addresses are read from it.
// Each wave waits for its own copies with an explicit vector-memory count: a wave
// issues the same number NOPS of copies per element, always in the same order, and loads
// complete in issue order, so element e's copies are complete once at most (AH-1)*NOPS
// of the wave's operations are outstanding.  The wave's stores count as well and
// can only make that wait longer.
//
// Per element, both waves pass three LDS-only barriers:
//   B1  inputs of e in ring slot e%AH (each wave waited for its own copies),
//       viscous residuals of the previous element handed over in LDS; wave 0
//       then completes that element's residual records
//   B2  nodal fields of e staged, slot e%AH read into registers (the copies
//       of element e+AH may start), previous element's records complete
//   B3  line derivatives of u and rho handed over: wave 0 forms them for the
//       convection terms, and wave 1 takes them for grad u and grad rho
//       instead of forming the same sums again
//
// What bounds it: 48.7 KB of LDS leave three workgroups per CU (k_rhs: 16 KB per wave,
// two waves per SIMD), and a cluster's flush waits for its node tables and state loads.
// Per stage at 262k elements: 1.60 ms and 0.28 ms for the gather over the surface nodes,
// against 0.64 and 0.37 ms in the node-ordered assembly.
template <int P, typename T, bool G16> struct SplitLDS {
    static constexpr int NN = (P + 1) * (P + 1) * (P + 1);
    static constexpr int AH = 2; // ring depth (elements in flight per block)
    // geometry, He then gpvol, copied in 64-lane rows of GW bytes per lane
    static constexpr int HE_BYTES = 9 * NN * (int)sizeof(T), GV_BYTES = NN * (int)sizeof(T);
    static constexpr int GW = G16 ? 16 : 4, GROW = 64 * GW;
    static constexpr int GROWS = (HE_BYTES + GV_BYTES + GROW - 1) / GROW, GEO = GROWS * GROW;
    // conserved fields rho, q1, q2, q3, E (FP64, node-major), then mu_e
    // mu_e(nelem,ngaus) is element-fastest: the 64 values of one element lie
    // nelem apart.  It is copied per run of RUN = 2 consecutive elements of the
    // cluster order (they pair up as e, e+1 on a box mesh), RUN values per node,
    // into one of three blocks, two runs ahead
    static constexpr int RUN = 2;
    static constexpr int ST = 5 * NN * 8;
    static constexpr int SLOT = GEO + ST;
    // connectivity rows: AH + 1 in use at a time
    static constexpr int CROWS = AH + 1, CROW = NN * 4;
    static constexpr int MUB = RUN * NN * (int)sizeof(T), MUBS = 3;
    static constexpr int MUB_AT = AH * SLOT + CROWS * CROW;
    static constexpr int BYTES = MUB_AT + MUBS * MUB;
    static constexpr int MU_OPS = (int)sizeof(T) / 4;
    static_assert(MUB == 256 * MU_OPS * RUN,
                  "one run's mu_e block in MU_OPS rows per element");
    // copies per element: wave 0 takes the connectivity row, the even
    // geometry rows and rho, q1, q2; wave 1 the odd rows, q3, E and mu_e
    static constexpr int NOPS0 = 1 + (GROWS + 1) / 2 + 6,
                         NOPS1 = GROWS / 2 + 4 + MU_OPS;
    static_assert(SLOT % 16 == 0, "ring slots must stay 16-byte aligned");
    static_assert(AH >= 2 && AH * NOPS0 <= 63 && AH * NOPS1 <= 63, "vmcnt range");
};

template <int P, typename T> struct SplitState {
    double cr, cq[3], cE;
    T mue;
};

// Copies of element e into the ring slot at LDS address slot and, by wave 0,
// the connectivity row of element ec to LDS address crow.  n0 and n1 are the
// global nodes of e at lexicographic (I fastest) positions lane/2 and
// 32 + lane/2: a 64-lane row of a field moves both 4-byte halves of 32 nodes,
// so the field lands as doubles in lexicographic node order, and on a mesh
// numbered along I each row reads 8 runs of p+1 consecutive nodes.
template <int P, typename T, bool G16, int ROLE>
__device__ __forceinline__ void split_issue(const RhsArgs<T> &A, unsigned slot, unsigned crow,
                                            int e, int ec, int n0, int n1, int lane)
{
    using L = SplitLDS<P, T, G16>;
    constexpr int NN = L::NN;
    const int hw = 4 * (lane & 1);
    if constexpr (ROLE == 0) dma_lds<4>(A.connecT + (size_t)ec * NN + lane, crow);
    const unsigned char *he = (const unsigned char *)(A.He + (size_t)e * 9 * NN);
    const unsigned char *gv = (const unsigned char *)(A.gpvol + (size_t)e * NN);
#pragma unroll
    for (int r = ROLE; r < L::GROWS; r += 2) {
        // lanes past the end of gpvol re-read its last GW bytes
        const int byte = r * L::GROW + lane * L::GW;
        const unsigned char *src =
            byte < L::HE_BYTES ? he + byte : gv + min(byte - L::HE_BYTES, L::GV_BYTES - L::GW);
        dma_lds<L::GW>(src, slot + r * L::GROW);
    }
    const size_t np = (size_t)A.npoin;
    const double *fld[5] = {A.cr, A.cq, A.cq + np, A.cq + 2 * np, A.cE};
    const unsigned st = slot + L::GEO;
#pragma unroll
    for (int f = ROLE == 0 ? 0 : 3; f < (ROLE == 0 ? 3 : 5); ++f) {
        dma_lds<4>((const char *)(fld[f] + n0) + hw, st + f * NN * 8);
        dma_lds<4>((const char *)(fld[f] + n1) + hw, st + f * NN * 8 + 256);
    }
}

// mu_e copies of one iteration: rows 2j and 2j+1 of
// the block of the run of elements e0, e1 (j = iteration within its run).
// The block is node-major and element-fastest: lane L moves half L&1 of
// mu_e(e_{(L/2)&1}, 16i + L/4) of row i.
template <typename T>
__device__ __forceinline__ void mu_issue2(const RhsArgs<T> &A, unsigned blk, int e0, int e1, int j,
                                          int lane)
{
    const int hw = 4 * (lane & 1), nd16 = lane >> 2;
    const int e = ((lane >> 1) & 1) ? e1 : e0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int i = 2 * j + h;
        dma_lds<4>((const char *)(A.mu_e + e + (size_t)A.nelem * (16 * i + nd16)) + hw, blk + i * 256);
    }
}

// reads ring slot sl into registers: He, gpvol and the conserved fields of node a (lexicographic position pa)
template <int P, typename T, bool G16>
__device__ __forceinline__ void split_read(const unsigned char *sl, int a, int pa,
                                           T He[3][3], T &vol, SplitState<P, T> &x)
{
    using L = SplitLDS<P, T, G16>;
    constexpr int NN = L::NN;
    const T *hp = (const T *)sl + 9 * a;
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int i = 0; i < 3; ++i) He[i][j] = hp[i + 3 * j];
    vol = ((const T *)sl)[9 * NN + a];
    const double *st = (const double *)(sl + L::GEO);
    x.cr = st[pa];
    x.cq[0] = st[NN + pa];
    x.cq[1] = st[2 * NN + pa];
    x.cq[2] = st[3 * NN + pa];
    x.cE = st[4 * NN + pa];
}

// The two-wave kernel.  The staged nodal fields and the viscous fluxes are
// node-major records, so one 16-byte LDS read returns two fields of a
// neighbour and the field offsets are immediates of the read instruction:
//   node record (10 values): u1 u2 | u3 rho | p H | T - | padding
//   flux record (18 values): for k = 1..3, G_k of (grad rho, grad T, tau u,
//                            tau_1., tau_2., tau_3.)
// Both operators are evaluated as k_rhs evaluates them (the FP64 stage's K and z
// coefficients, the same sums in the same order; only the conductivity takes Cp/Pr as
// one factor), so that this assembly and the node-ordered one differ by the order of a
// surface node's terms and that rounding.
// The block walks element clusters, one after the other; the viscous wave adds each
// element's residual records into an LDS accumulator per cluster-local node, and after
// a cluster's last element finishes its interior nodes (mass inverse and
// stage combine, as k_gather_update) and stores one partial record per
// surface node.
template <int P, typename T, bool G16>
__global__ __launch_bounds__(128, 2) void k_rhs_split(RhsArgs<T> A)
{
    using L = SplitLDS<P, T, G16>;
    static_assert(sizeof(T) == 8 && P == 3, "cluster assembly: FP64, p=3");
    using V2 = T __attribute__((ext_vector_type(2)));
    // node records of REC values: 80 bytes, an odd multiple of 16, so that 16
    // lanes reading 16 consecutive records with 16-byte reads hit distinct
    // banks; 144-byte flux records
    constexpr int NN = L::NN, REC = 10, GREC = 18, AH = L::AH;
    // s2 holds, in turn: the viscous flux records (GREC values per node) and
    // the handed-over viscous residuals (3 pairs per node), then the dense
    // residual records (RW values per node) followed by the line derivatives
    // of u and rho (6 pairs per node) from DREC on
    constexpr int RW = 5; // values per residual record
    constexpr int DREC = RW * NN / 2;
    static_assert(DREC + 6 * NN <= 64 * GREC / 2, "derivative records fit in s2");
    static_assert(NN == 64, "one lane per node");
    __shared__ V2 s1[64 * REC / 2]; // records of REC values as pairs
    __shared__ V2 s2[64 * GREC / 2];
    __shared__ __attribute__((aligned(16))) unsigned char ring[L::BYTES];
    const unsigned ring_lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)ring;
    // the block's element order and local-node ranges, the
    // local-index rows of the last AH + 1 elements, the accumulator
    constexpr int G = kClusterG, CMAX = kClusterBlockMax, CR = AH + 1;
    __shared__ int cel_s[CMAX * G];
    __shared__ int cb_s[2 * CMAX];
    __shared__ __attribute__((aligned(16))) int cloc_s[CR * 64];
    __shared__ double acc_s[5 * kClusterLMax];
    const unsigned cloc_lds =
        (unsigned)(uintptr_t)(__attribute__((address_space(3))) int *)cloc_s;

    const int role = threadIdx.x >> 6; // 0: convection, 1: viscous (wave-uniform)
    const int lane = threadIdx.x & 63;
    const bool visc = role == 1;

    constexpr int RUN = L::RUN, RSH = 1;
    // over clusters
    const ElemRange er = elem_range(A.ncl);
    if (er.begin >= er.end) return;
    const int nunits = (er.end - er.begin + er.stride - 1) / er.stride;
    const int nit = G * nunits;
    // a padding slot (-1) of a cluster evaluates its first element again
    // and adds nothing
    for (int i = threadIdx.x; i < nunits * G; i += 128) {
        const long c = er.begin + (long)(i / G) * er.stride;
        cel_s[i] = A.cel[c * G + i % G];
    }
    for (int i = threadIdx.x; i < nunits; i += 128) {
        const long c = er.begin + (long)i * er.stride;
        cb_s[2 * i] = A.cnb[c];
        cb_s[2 * i + 1] = A.cnb[c + 1];
    }
    for (int i = threadIdx.x; i < 5 * kClusterLMax; i += 128) acc_s[i] = 0.0;
    __syncthreads();
    // element of iteration t.  Past the block's last element the copies, which stay
    // unconditional, repeat that element.
    auto elem_of = [&](int t) {
        const int i = min(t, nit - 1);
        const int e = cel_s[i];
        return e >= 0 ? e : cel_s[i - i % G];
    };
    // mu_e blocks: iteration t (t >= -2 RUN) copies its share of the
    // block of run t/RUN + 2 (floor); the block of run r is read from
    // iteration RUN r on
    auto mu_at = [&](int t) {
        const int r = (t >> RSH) + 2;
        const unsigned blk = ring_lds + L::MUB_AT + (r % 3) * L::MUB;
        mu_issue2<T>(A, blk, elem_of(r * RUN), elem_of(r * RUN + 1), t & (RUN - 1), lane);
    };
    auto mu_read = [&](int t, int node) {
        return ((const T *)(ring + L::MUB_AT + ((t >> RSH) % 3) * L::MUB))[node * RUN + (t & (RUN - 1))];
    };
    // the local-index row of iteration t's element, copied by
    // the viscous wave with its share of that element's inputs
    auto cloc_issue = [&](int t) {
        const int i = min(t, nit - 1);
        const long c = er.begin + (long)(i / G) * er.stride;
        dma_lds<4>(A.cloc + ((size_t)c * G + i % G) * NN + lane, cloc_lds + (t % CR) * 256);
    };
    auto slot_of = [&](int t) { return (t % AH) * L::SLOT; };
    auto crow_of = [&](int t) { return AH * L::SLOT + (t % L::CROWS) * L::CROW; };
    const int nd = lane >> 1;

    // Lane L evaluates the node a at lexicographic position L (I fastest);
    // the LDS records are kept in that order.  Along every line direction
    // the 16 lanes of an LDS access phase then read 16 distinct records
    // (a permutation of 16 consecutive ones).  ia0, ia1: the nodes at
    // lexicographic positions nd and 32 + nd.
    auto lex = [&](int r) { return min(max(A.perm[r], 0), NN - 1); };
    int a, ia0, ia1;
    {
        int *inv = (int *)s1;
        if (role == 0) inv[lex(lane)] = lane;
        lds_barrier();
        a = min(max(inv[lane], 0), NN - 1);
        ia0 = min(max(inv[nd], 0), NN - 1);
        ia1 = min(max(inv[32 + nd], 0), NN - 1);
        lds_barrier();
    }
    const int pa = lane;
    LineTab<P, T> lt;
    build_linetab<P, T>(a, A.dl, A.inv, A.gI, A.gJ, A.gK, lt);
    // neighbour records (element offsets into s1)
    int nb[3][P];
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int o = 0; o < P; ++o) nb[k][o] = lex(lt.off[k][o]) * REC;
    const int own = pa * REC;

    // the connectivity of the first AH elements, then the first AH elements
    // in the ring in the order of the main loop
    if (role == 0)
        for (int t = 0; t < AH; ++t)
            dma_lds<4>(A.connecT + (size_t)elem_of(t) * NN + lane, ring_lds + crow_of(t));
    else
        for (int t = -2 * RUN; t < -AH; ++t) mu_at(t);
    wait_vm<0>();
    lds_barrier();
    for (int t = 0; t < AH; ++t) {
        const int *c = (const int *)(ring + crow_of(t));
        const int n0 = c[ia0], n1 = c[ia1];
        if (visc) {
            split_issue<P, T, G16, 1>(A, ring_lds + slot_of(t), ring_lds + crow_of(t + AH), elem_of(t),
                                      elem_of(t + AH), n0, n1, lane);
            mu_at(t - AH);
            cloc_issue(t);
        } else
            split_issue<P, T, G16, 0>(A, ring_lds + slot_of(t), ring_lds + crow_of(t + AH), elem_of(t),
                                      elem_of(t + AH), n0, n1, lane);
        lds_barrier(); // the row read here is rewritten in a later pass
    }
    SplitState<P, T> cur;

    auto prim = [&](const SplitState<P, T> &c, double &r, double ud[3], double &pd, double &hd,
                    double &Td, double &umag) {
        r = c.cr;
        const double ri = 1.0 / r;
        umag = 0.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            ud[d] = c.cq[d] * ri;
            umag += ud[d] * ud[d];
        }
        const double eint = c.cE * ri - 0.5 * umag;
        pd = r * (A.gamma - 1.0) * eint;
        hd = (A.gamma / (A.gamma - 1.0)) * pd * ri;
        Td = pd * ri / A.Rgas;
    };
        // indices are even value offsets into the records
#define LD1(i) (s1[(i) >> 1].x)
#define LD2(i) (s1[(i) >> 1])
#define GL2(i) (s2[(i) >> 1])

    if (!visc) {
        // ======================= convection wave
        // convection residuals (times gpvol) of the previous element
        T pend[5] = {0, 0, 0, 0, 0};
        // its records: pend plus the viscous residuals handed over in s2, as
        // dense records in lexicographic node order over the same LDS (all
        // lanes read before any writes; a padded record is exactly the slot
        // the lane read its handover from); the viscous wave stores them
        auto finish = [&]() {
            const V2 h01 = s2[3 * pa], h23 = s2[3 * pa + 1], h4 = s2[3 * pa + 2];
            T *d = (T *)s2 + RW * pa;
            d[0] = pend[0] + h01.x;
            d[1] = pend[1] + h01.y;
            d[2] = pend[2] + h23.x;
            d[3] = pend[3] + h23.y;
            d[4] = pend[4] + h4.x;
        };
        for (int t = 0; t < nit; ++t) {
            wait_vm<(AH - 1) * L::NOPS0>();
            lds_barrier(); // B1
            if (t != 0) finish();
            T He[3][3], vol;
            split_read<P, T, G16>(ring + slot_of(t), a, pa, He, vol, cur);
            T rho, u[3], p, H;
            {
                double r, ud[3], pd, hd, Td, umag;
                prim(cur, r, ud, pd, hd, Td, umag);
                rho = T(r);
#pragma unroll
                for (int d = 0; d < 3; ++d) u[d] = T(ud[d]);
                p = T(pd - A.p_ref);
                H = T(hd + 0.5 * umag);
                s1[(own + 0) >> 1] = V2{u[0], u[1]};
                s1[(own + 2) >> 1] = V2{u[2], rho};
                s1[(own + 4) >> 1] = V2{p, H};
            }
            lds_barrier(); // B2
            {
                const int *c = (const int *)(ring + crow_of(t + AH));
                split_issue<P, T, G16, 0>(A, ring_lds + slot_of(t), ring_lds + crow_of(t + 2 * AH),
                                          elem_of(t + AH), elem_of(t + 2 * AH), c[ia0], c[ia1], lane);
            }

            T Rq[3] = {0, 0, 0}, Re = 0;
            T Ut[3], divU = 0;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                Ut[k] = He[0][k] * u[0] + He[1][k] * u[1] + He[2][k] * u[2];
                divU += lt.ds[k] * Ut[k];
            }
            // velocity and density lines: the coefficients K_k(m), the momentum
            // sums, div u, div q + u.grad rho, and the line derivatives for the
            // viscous wave
            const T a0 = divU;
            T s = T(2) * rho * a0, Kx[3][P];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const T c0 = lt.ds[k];
                T du[3], dr = c0 * rho, rq[3] = {0, 0, 0}, dvu = 0, dvq = 0;
#pragma unroll
                for (int i = 0; i < 3; ++i) du[i] = c0 * u[i];
#pragma unroll
                for (int o = 0; o < P; ++o) {
                    const T c = lt.d[k][o];
                    const V2 x01 = LD2(nb[k][o] + 0), x2r = LD2(nb[k][o] + 2);
                    dr += c * x2r.y;
                    const T ut = He[0][k] * x01.x + He[1][k] * x01.y + He[2][k] * x2r.x;
                    const T z = c * (Ut[k] + ut), K = z * (rho + x2r.y);
                    Kx[k][o] = K;
                    dvu += c * ut;
                    dvq += z * x2r.y;
                    rq[0] += K * x01.x;
                    rq[1] += K * x01.y;
                    rq[2] += K * x2r.x;
                    du[0] += c * x01.x;
                    du[1] += c * x01.y;
                    du[2] += c * x2r.x;
                }
#pragma unroll
                for (int i = 0; i < 3; ++i) Rq[i] += rq[i];
                divU += dvu;
                s += dvq;
                s2[DREC + 6 * pa + 2 * k] = V2{du[0], du[1]};
                s2[DREC + 6 * pa + 2 * k + 1] = V2{du[2], dr};
            }
            lds_barrier(); // B3
            // pressure gradient and the enthalpy's sum
            T dp[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                T re = 0;
                dp[k] = lt.ds[k] * p;
#pragma unroll
                for (int o = 0; o < P; ++o) {
                    const V2 x = LD2(nb[k][o] + 4);
                    re += Kx[k][o] * x.y;
                    dp[k] += lt.d[k][o] * x.x;
                }
                Re += re;
            }
            const T B = s + rho * (divU + T(4) * a0);
            pend[0] = vol * (T(0.5) * (s + rho * divU));
#pragma unroll
            for (int i = 0; i < 3; ++i)
                pend[1 + i] = vol * (T(0.25) * (Rq[i] + u[i] * B) +
                                     (He[i][0] * dp[0] + He[i][1] * dp[1] + He[i][2] * dp[2]));
            pend[4] = vol * (T(0.25) * (Re + H * B));
        }
        // the last element's records
        lds_barrier();
        finish();
        lds_barrier();
    } else {
        // ======================= viscous wave
        const T cp_pr = A.Cp / A.Pr;
        T tt[3][P];
        {
            const int own3[3] = {min(max(A.gI[a] - 1, 0), P), min(max(A.gJ[a] - 1, 0), P),
                                 min(max(A.gK[a] - 1, 0), P)};
#pragma unroll
            for (int k = 0; k < 3; ++k)
#pragma unroll
                for (int o = 0; o < P; ++o) tt[k][o] = A.dl[lt.off[k][o] + NN * (k + 3 * own3[k])];
        }
        int gnb[3][P];
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int o = 0; o < P; ++o) gnb[k][o] = lex(lt.off[k][o]) * GREC + 6 * k;
        // adds iteration tt's dense records (s2, lexicographic
        // node order) into the accumulator at the element's local nodes (64
        // distinct local nodes per element: no two lanes collide)
        auto cl_accumulate = [&](int tt) {
            const int i = min(tt, nit - 1);
            if (cel_s[i] < 0) return; // padding slot
            const int sl = min(max(cloc_s[(tt % CR) * 64 + lane], 0), kClusterLMax - 1);
            const T *d = (const T *)s2 + RW * lane;
            double *ac = acc_s + 5 * sl;
#pragma unroll
            for (int f = 0; f < 5; ++f) ac[f] += (double)d[f];
        };
        // after the last element of the cluster of iteration tt:
        // interior working nodes get R = fact * sum * invMl and the stage
        // combine (k_gather_update's arithmetic; the sum runs over the same
        // elements in the same ascending order), surface working nodes one
        // partial record; the accumulator is cleared for the next cluster
        auto cl_flush = [&](int tt) {
            const int k = min(tt, nit - 1) / G;
            const int base = cb_s[2 * k], lim = cb_s[2 * k + 1];
            const size_t np = (size_t)A.npoin;
            for (int l = base + lane; l < lim; l += 64) {
                double v[5];
                double *ac = acc_s + 5 * (l - base);
#pragma unroll
                for (int f = 0; f < 5; ++f) {
                    v[f] = ac[f];
                    ac[f] = 0.0;
                }
                const int kind = A.ckind[l];
                if (kind == 1) {
                    double *r = A.rec + 5 * (size_t)l;
#pragma unroll
                    for (int f = 0; f < 5; ++f) r[f] = v[f];
                } else if (kind == 0) {
                    const size_t n = (size_t)A.cnode[l];
                    const size_t k3[5] = {n, n, n + np, n + 2 * np, n};
                    const double *y1v[5] = {A.y1r, A.y1q, A.y1q, A.y1q, A.y1E};
                    double *yv[5] = {A.yr, A.yq, A.yq, A.yq, A.yE};
                    double *rv[5] = {A.Rm, A.Rq, A.Rq, A.Rq, A.Re};
                    double *xv[5] = {A.nxr, A.nxq, A.nxq, A.nxq, A.nxE};
                    const double m = A.invMl[n];
                    double b[5], y[5];
#pragma unroll
                    for (int f = 0; f < 5; ++f) {
                        b[f] = A.rd1 ? y1v[f][k3[f]] : 0.0;
                        y[f] = A.rdy ? yv[f][k3[f]] : 0.0;
                    }
#pragma unroll
                    for (int f = 0; f < 5; ++f) {
                        const double r = (A.fact * v[f]) * m;
                        const double z = A.lam1 * b[f] + A.lams * y[f] + A.gdt * r;
                        yv[f][k3[f]] = z;
                        if (A.nxr) {
                            const double zero = 0.0, nls = 0.0;
                            xv[f][k3[f]] = A.nx_l1 * z + nls * zero + A.nx_gdt * r;
                        }
                        if (A.Rm) rv[f][k3[f]] = r;
                    }
                }
            }
        };
        for (int t = 0; t < nit; ++t) {
            wait_vm<(AH - 1) * (L::NOPS1 + 1)>();
            lds_barrier(); // B1
            T He[3][3], vol;
            split_read<P, T, G16>(ring + slot_of(t), a, pa, He, vol, cur);
            cur.mue = mu_read(t, a);
            T rho, u[3], Tk, muf;
            const T mue = cur.mue;
            {
                double r, ud[3], pd, hd, Td, umag;
                prim(cur, r, ud, pd, hd, Td, umag);
                rho = T(r);
#pragma unroll
                for (int d = 0; d < 3; ++d) u[d] = T(ud[d]);
                Tk = T(Td);
                const double mfe = A.mu_factor_e ? A.mu_factor_e[elem_of(t)] : A.mu_factor;
                muf = T(sutherland<double>(mfe, Td));
                s1[(own + 6) >> 1] = V2{Tk, T(0)};
            }
            lds_barrier(); // B2
            // the previous element's records go into the
            // accumulator before its local-index row is overwritten below
            if (t != 0) cl_accumulate(t - 1);
            {
                const int *c = (const int *)(ring + crow_of(t + AH));
                split_issue<P, T, G16, 1>(A, ring_lds + slot_of(t), ring_lds + crow_of(t + 2 * AH),
                                          elem_of(t + AH), elem_of(t + 2 * AH), c[ia0], c[ia1], lane);
                mu_at(t);
                cloc_issue(t + AH);
            }
            if (t != 0 && t % G == 0) cl_flush(t - 1);
            // grad T from the T lines; grad u and grad rho from the line
            // derivatives handed over by the convection wave
            T dT[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                T vt = lt.ds[k] * Tk;
#pragma unroll
                for (int o = 0; o < P; ++o) vt += lt.d[k][o] * LD1(nb[k][o] + 6);
                dT[k] = vt;
            }
            // formed here, while the convection wave is on its lines, and with one
            // division: at the end of the element, where they are used, three divisions
            // held up both waves (element kernel at 262k elements 1684 -> 1595 us,
            // 1,728 elements 340 -> 311 us)
            T nu_e = A.c_rho * mue / rho;
            T kappa = (muf + A.c_ener * mue) * cp_pr;
            pin(nu_e);
            pin(kappa);
            lds_barrier(); // B3
            T gU[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
            T dr[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const V2 d01 = s2[DREC + 6 * pa + 2 * k], d2r = s2[DREC + 6 * pa + 2 * k + 1];
                const T du[3] = {d01.x, d01.y, d2r.x};
                dr[k] = d2r.y;
#pragma unroll
                for (int i = 0; i < 3; ++i)
#pragma unroll
                    for (int j = 0; j < 3; ++j) gU[i][j] += He[j][k] * du[i];
            }
            T gR[3], gt[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                gR[i] = He[i][0] * dr[0] + He[i][1] * dr[1] + He[i][2] * dr[2];
                gt[i] = He[i][0] * dT[0] + He[i][1] * dT[1] + He[i][2] * dT[2];
            }
            // contravariant fluxes G_k(F) = gpvol sum_d He(d,k) F_d into the flux record
            const T mut = muf + mue;
            const T divU = gU[0][0] + gU[1][1] + gU[2][2];
            const T tdiv = muf * T(2.0 / 3.0) * divU;
            T tau[3][3];
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int j = 0; j < 3; ++j) tau[i][j] = mut * (gU[i][j] + gU[j][i]);
#pragma unroll
            for (int i = 0; i < 3; ++i) tau[i][i] -= tdiv;
            const int g = pa * GREC;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const T h0 = vol * He[0][k], h1 = vol * He[1][k], h2 = vol * He[2][k];
                T gr[3], tuk = 0;
#pragma unroll
                for (int r = 0; r < 3; ++r) {
                    gr[r] = h0 * tau[r][0] + h1 * tau[r][1] + h2 * tau[r][2];
                    tuk += gr[r] * u[r]; // tau is symmetric: contravariant (tau u)_k
                }
                s2[(g + 6 * k + 0) >> 1] = V2{h0 * gR[0] + h1 * gR[1] + h2 * gR[2],
                                            h0 * gt[0] + h1 * gt[1] + h2 * gt[2]};
                s2[(g + 6 * k + 2) >> 1] = V2{tuk, gr[0]};
                s2[(g + 6 * k + 4) >> 1] = V2{gr[1], gr[2]};
            }
            // this wave alone reads s2 next: its LDS instructions execute in order
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
            // pass 2: weak divergence sum_k sum_b dl(b,k,I_k(a)) G_k(F)(b)
            T W6[6] = {0, 0, 0, 0, 0, 0};
            {
                const int g = pa * GREC;
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    const V2 o01 = GL2(g + 6 * k), o23 = GL2(g + 6 * k + 2), o45 = GL2(g + 6 * k + 4);
                    const T own6[6] = {o01.x, o01.y, o23.x, o23.y, o45.x, o45.y};
#pragma unroll
                    for (int f = 0; f < 6; ++f) W6[f] += lt.ds[k] * own6[f];
                }
#pragma unroll
                for (int k = 0; k < 3; ++k)
#pragma unroll
                    for (int o = 0; o < P; ++o) {
                        const T c = tt[k][o];
                        const V2 x01 = GL2(gnb[k][o]), x23 = GL2(gnb[k][o] + 2), x45 = GL2(gnb[k][o] + 4);
                        W6[0] += c * x01.x;
                        W6[1] += c * x01.y;
                        W6[2] += c * x23.x;
                        W6[3] += c * x23.y;
                        W6[4] += c * x45.x;
                        W6[5] += c * x45.y;
                    }
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
            s2[3 * pa] = V2{nu_e * W6[0], W6[3]};
            s2[3 * pa + 1] = V2{W6[4], W6[5]};
            s2[3 * pa + 2] = V2{W6[2] + kappa * W6[1], T(0)};
        }
        // the last element's records, completed by the convection wave
        lds_barrier();
        lds_barrier();
        cl_accumulate(nit - 1);
        cl_flush(nit - 1);
    }
    // no copy may still be writing this block's LDS when it retires
    wait_vm<0>();
#undef LD1
#undef LD2
#undef GL2
}

// Launches the operators' element kernel.  bpc: the stage's elem_blocks_per_cu setting
// (16: the kernel's own launch shape; others scale the units a block takes).
template <int P, typename T, bool CONV, int VISC, bool CONS>
static void launch_rhs_p(sodhip_ctx ctx, RhsArgs<T> A, int bpc)
{
    const UnitShape us = unit_shape<P, T>(ctx, A.nelem, bpc);
    A.run = us.run;
    A.wide = us.wide;
    k_rhs<P, T, CONV, VISC, CONS><<<us.grid, EP<P, T>::NTB, 0, ctx->stream>>>(A);
}

template <typename T>
static int launch_rhs(sodhip_ctx ctx, int porder, bool conv, bool diff, bool cons,
                      const RhsArgs<T> &A0, int bpc = 16, int geo16 = 1)
{
    RhsArgs<T> A = A0;
    // 16-byte geometry copies start from 16-byte boundaries of the arrays
    A.geo16 = geo16 && ((uintptr_t)A.He % 16 == 0) && ((uintptr_t)A.gpvol % 16 == 0);
#define SODHIP_RHS_CASE(PP)                                                                \
    case PP:                                                                               \
        if (conv && diff && cons)                                                          \
            launch_rhs_p<PP, T, true, 1, true>(ctx, A, bpc);                            \
        else if (conv && !diff && !cons)                                                   \
            launch_rhs_p<PP, T, true, 0, false>(ctx, A, bpc);                          \
        else if (!conv && diff && !cons)                                                   \
            launch_rhs_p<PP, T, false, 1, false>(ctx, A, bpc);                          \
        else                                                                               \
            return set_error(SODHIP_ERR_UNSUPPORTED, "unsupported operator combination");  \
        break;
    switch (porder) {
        SODHIP_RHS_CASE(2)
        SODHIP_RHS_CASE(3)
        SODHIP_RHS_CASE(4)
    default:
        return set_error(SODHIP_ERR_UNSUPPORTED, "porder %d not supported (2..4)", porder);
    }
#undef SODHIP_RHS_CASE
    SODHIP_TRY_HIP(hipGetLastError());
    return SODHIP_OK;
}

template <typename TS, typename TR>
static int launch_gather(sodhip_ctx ctx, const MeshCache *m, const TS *scr, int nf,
                         TR *R0, TR *R1, TR *R2, TR *R3, TR *R4, int init, TR fact)
{
    const int bs = 256;
    const int grid = ((m->npoin + bs - 1) / bs + 7) / 8 * 8;
#define SODHIP_GATHER(NFV)                                                                     \
    k_gather<TS, TR, NFV><<<grid, bs, 0, ctx->stream>>>(m->npoin, m->row, m->src, scr, R0, R1,  \
                                                        R2, R3, R4, init, fact)
    switch (nf) {
    case 1: SODHIP_GATHER(1); break;
    case 3: SODHIP_GATHER(3); break;
    case 4: SODHIP_GATHER(4); break;
    case 5: SODHIP_GATHER(5); break;
    default: return set_error(SODHIP_ERR_UNSUPPORTED, "gather of %d fields", nf);
    }
#undef SODHIP_GATHER
    SODHIP_TRY_HIP(hipGetLastError());
    return SODHIP_OK;
}

template <typename T>
static int check_common(sodhip_ctx ctx, int porder, int nelem, int npoin, const int *connec)
{
    SODHIP_REQUIRE(ctx, "null context");
    SODHIP_REQUIRE(porder >= 2 && porder <= kMaxP, "porder %d not supported (2..4)", porder);
    SODHIP_REQUIRE(nelem > 0 && npoin > 0 && connec, "invalid mesh arguments");
    return SODHIP_OK;
}

template <typename T>
static int full_convec(sodhip_ctx ctx, int porder, int nelem, int npoin, const int *connec,
                       const T *He, const T *gpvol, const T *dl, const int *inv, const int *gI,
                       const int *gJ, const int *gK, const T *u, const T *q, const T *rho,
                       const T *pr, const T *E, T *Rmass, T *Rmom, T *Rener, int initialize,
                       T fact)
{
    int rc = check_common<T>(ctx, porder, nelem, npoin, connec);
    if (rc) return rc;
    SODHIP_REQUIRE(He && gpvol && dl && inv && gI && gJ && gK && u && q && rho && pr && E &&
                       Rmass && Rmom && Rener,
                   "null array argument");
    SODHIP_TRY_HIP(hipSetDevice(ctx->device));
    MeshCache *m = nullptr;
    if ((rc = get_mesh(ctx, porder, nelem, npoin, connec, &m))) return rc;
    const size_t EN = (size_t)nelem * nnode_of(porder);
    if ((rc = ensure_buf(ctx->scratch, 5 * EN * sizeof(T)))) return rc;
    RhsArgs<T> A{};
    A.nelem = nelem;
    A.npoin = npoin;
    A.connecT = m->connecT;
    A.perm = m->perm;
    A.He = He;
    A.gpvol = gpvol;
    A.dl = dl;
    A.inv = inv;
    A.u = u;
    A.q = q;
    A.rho = rho;
    A.pr = pr;
    A.E = E;
    A.out = (T *)ctx->scratch.ptr;
    int tok = prof_begin(ctx, 0);
    rc = launch_rhs<T>(ctx, porder, true, false, false, A);
    prof_end(ctx, tok);
    if (rc) return rc;
    tok = prof_begin(ctx, 1);
    rc = launch_gather<T, T>(ctx, m, A.out, 5, Rmass, Rmom, Rmom + npoin,
                             Rmom + 2 * (size_t)npoin, Rener, initialize, fact);
    prof_end(ctx, tok);
    return rc;
}

template <typename T>
static int full_diffusion(sodhip_ctx ctx, int porder, int nelem, int npoin, const int *connec,
                          const T *He, const T *gpvol, const T *dl, const int *inv, const int *gI,
                          const int *gJ, const int *gK, T Cp, T Pr, const T *rho_n, const T *rho,
                          const T *u, const T *Tem, const T *mu_fluid, const T *mu_e,
                          const T *mu_sgs, T c_rho, T c_ener, T *Rmass, T *Rmom, T *Rener,
                          int initialize, T fact)
{
    int rc = check_common<T>(ctx, porder, nelem, npoin, connec);
    if (rc) return rc;
    SODHIP_REQUIRE(He && gpvol && dl && inv && gI && gJ && gK && rho_n && rho && u && Tem &&
                       mu_fluid && mu_e && Rmass && Rmom && Rener,
                   "null array argument");
    SODHIP_TRY_HIP(hipSetDevice(ctx->device));
    MeshCache *m = nullptr;
    if ((rc = get_mesh(ctx, porder, nelem, npoin, connec, &m))) return rc;
    const size_t EN = (size_t)nelem * nnode_of(porder);
    if ((rc = ensure_buf(ctx->scratch, 5 * EN * sizeof(T)))) return rc;
    RhsArgs<T> A{};
    A.nelem = nelem;
    A.npoin = npoin;
    A.connecT = m->connecT;
    A.perm = m->perm;
    A.He = He;
    A.gpvol = gpvol;
    A.dl = dl;
    A.inv = inv;
    A.rho = rho;
    A.u = u;
    A.rho_n = rho_n;
    A.Tem = Tem;
    A.mu_fluid = mu_fluid;
    A.mu_e = mu_e;
    A.mu_sgs = mu_sgs;
    A.Cp = Cp;
    A.Pr = Pr;
    A.c_rho = c_rho;
    A.c_ener = c_ener;
    A.out = (T *)ctx->scratch.ptr;
    int tok = prof_begin(ctx, 0);
    rc = launch_rhs<T>(ctx, porder, false, true, false, A);
    prof_end(ctx, tok);
    if (rc) return rc;
    tok = prof_begin(ctx, 1);
    rc = launch_gather<T, T>(ctx, m, A.out, 5, Rmass, Rmom, Rmom + npoin,
                             Rmom + 2 * (size_t)npoin, Rener, initialize, fact);
    prof_end(ctx, tok);
    return rc;
}

// Fused RHS used by the stage driver (ops_stage.hip): convection + viscous
// operator from the conserved FP64 state; writes element partials only.
// values per record of rhs_fused_elements' output (operator precision 8 or 4)
int fused_record_width(int porder, int op_bytes)
{
    return op_bytes == 4 && porder == 3 ? stage_rw<3, float>() : 5;
}

template <typename T>
int rhs_fused_elements(sodhip_ctx ctx, int porder, const MeshCache *m, const T *He,
                       const T *gpvol, const T *dl, const int *inv, const double *rho,
                       const double *q, const double *E, const T *mu_e, double gamma, double Rgas, double Cp, double Pr,
                       double mu_factor, const double *mu_factor_e, double c_rho, double c_ener,
                       double p_ref, T *out)
{
    RhsArgs<T> A{};
    A.nelem = m->nelem;
    A.npoin = m->npoin;
    A.connecT = m->connecT;
    A.perm = m->perm;
    A.He = He;
    A.gpvol = gpvol;
    A.dl = dl;
    A.inv = inv;
    A.cr = rho;
    A.cq = q;
    A.cE = E;
    A.mu_e = mu_e;
    A.gamma = gamma;
    A.Rgas = Rgas;
    A.mu_factor = mu_factor;
    A.mu_factor_e = mu_factor_e;
    A.p_ref = p_ref;
    A.Cp = T(Cp);
    A.Pr = T(Pr);
    A.c_rho = T(c_rho);
    A.c_ener = T(c_ener);
    A.out = out;
    int tok = prof_begin(ctx, 0);
    const int rc = launch_rhs<T>(ctx, porder, true, true, true, A, ctx->stage_bpc,
                                 ctx->stage_geo16);
    prof_end(ctx, tok);
    return rc;
}
int rhs_cluster_stage(sodhip_ctx ctx, const MeshCache *m, const ClusterTables *cl,
                      const double *He, const double *gpvol, const double *dl, const int *inv,
                      const int *gI, const int *gJ, const int *gK, const double *mu_e,
                      double gamma, double Rgas, double Cp, double Pr, double mu_factor,
                      const double *mu_factor_e, double c_rho, double c_ener, double p_ref,
                      const double *invMl, double fact, double dt, double lam1, double lams,
                      double gam, const double *rho1, const double *q1, const double *E1,
                      double *rho, double *q, double *E, double *Rmass, double *Rmom,
                      double *Rener, const NextStage *next, const double *const st[3],
                      double *rec)
{
    using T = double;
    RhsArgs<T> A{};
    A.nelem = m->nelem;
    A.npoin = m->npoin;
    A.connecT = m->connecT;
    A.perm = m->perm;
    A.He = He;
    A.gpvol = gpvol;
    A.dl = dl;
    A.inv = inv;
    A.gI = gI;
    A.gJ = gJ;
    A.gK = gK;
    A.cr = st[0];
    A.cq = st[1];
    A.cE = st[2];
    A.mu_e = mu_e;
    A.gamma = gamma;
    A.Rgas = Rgas;
    A.mu_factor = mu_factor;
    A.mu_factor_e = mu_factor_e;
    A.p_ref = p_ref;
    A.Cp = Cp;
    A.Pr = Pr;
    A.c_rho = c_rho;
    A.c_ener = c_ener;
    A.out = nullptr;
    A.cel = cl->cel;
    A.cloc = cl->cloc;
    A.cnb = cl->cnb;
    A.cnode = cl->cnode;
    A.ckind = cl->ckind;
    A.ncl = cl->ncl;
    A.rec = rec;
    A.invMl = invMl;
    A.fact = fact;
    A.lam1 = lam1;
    A.lams = lams;
    A.gdt = gam * dt;
    A.rd1 = lam1 != 0.0;
    A.rdy = lams != 0.0;
    A.y1r = rho1;
    A.y1q = q1;
    A.y1E = E1;
    A.yr = rho;
    A.yq = q;
    A.yE = E;
    A.Rm = Rmass;
    A.Rq = Rmom;
    A.Re = Rener;
    if (next) {
        A.nx_l1 = next->nl1;
        A.nx_gdt = next->ngdt;
        A.nxr = next->rho;
        A.nxq = next->q;
        A.nxE = next->E;
    }
    A.geo16 = ((uintptr_t)He % 16 == 0) && ((uintptr_t)gpvol % 16 == 0);
    // XCD-aware: every XCD's eighth of the clusters split over its blocks,
    // at most kClusterBlockMax clusters per block
    const long chunk = ((long)cl->ncl + 7) / 8;
    const long per = std::max<long>((chunk + kClusterBlockMax - 1) / kClusterBlockMax, 1);
    const int grid = (int)(8 * per);
    int tok = prof_begin(ctx, 0);
    if (A.geo16)
        k_rhs_split<3, T, true><<<grid, 128, 0, ctx->stream>>>(A);
    else
        k_rhs_split<3, T, false><<<grid, 128, 0, ctx->stream>>>(A);
    prof_end(ctx, tok);
    SODHIP_TRY_HIP(hipGetLastError());
    return SODHIP_OK;
}

// The LPS operators' element kernels (LpsArgs, common.hpp): the fused stage's
// convection and stabilised viscous operator from the conserved state (`stage`),
// the drop-in stabilised operator, or the projections' records.
int lps_elements(sodhip_ctx ctx, int porder, const MeshCache *m, const LpsArgs &L, LpsKernel what)
{
    RhsArgs<double> A{};
    A.nelem = m->nelem;
    A.npoin = m->npoin;
    A.connecT = m->connecT;
    A.perm = m->perm;
    A.He = L.He;
    A.gpvol = L.gpvol;
    A.dl = L.dl;
    A.inv = L.inv;
    A.rho = L.rho;
    A.u = L.u;
    A.Tem = L.Tem;
    A.rho_n = L.rho_n;
    A.mu_fluid = L.mu_fluid;
    A.mu_e = L.mu_e;
    A.mu_sgs = L.mu_sgs;
    A.cr = L.cr;
    A.cq = L.cq;
    A.cE = L.cE;
    A.gamma = L.gamma;
    A.Rgas = L.Rgas;
    A.mu_factor = L.mu_factor;
    A.Cp = L.Cp;
    A.Pr = L.Pr;
    A.c_rho = L.c_rho;
    A.c_ener = L.c_ener;
    A.c_lps = L.c_lps;
    A.tau = L.tau;
    A.prj = L.prj;
    A.pMass = L.pMass;
    A.pEner = L.pEner;
    A.pMX = L.pMX;
    A.pMY = L.pMY;
    A.pMZ = L.pMZ;
    A.out = L.out;
    A.geo16 = (what != LpsKernel::stage || ctx->stage_geo16) && ((uintptr_t)A.He % 16 == 0) &&
              ((uintptr_t)A.gpvol % 16 == 0);
    const int bpc = what == LpsKernel::stage ? ctx->stage_bpc : 16;
#define SODHIP_LPS_CASE(PP)                                                                \
    case PP:                                                                               \
        if (what == LpsKernel::stage)                                                      \
            launch_rhs_p<PP, double, true, 2, true>(ctx, A, bpc);                          \
        else if (what == LpsKernel::stab)                                                  \
            launch_rhs_p<PP, double, false, 2, false>(ctx, A, bpc);                        \
        else                                                                               \
            launch_rhs_p<PP, double, false, 3, false>(ctx, A, bpc);                        \
        break;
    switch (porder) {
        SODHIP_LPS_CASE(2)
        SODHIP_LPS_CASE(3)
        SODHIP_LPS_CASE(4)
    default:
        return set_error(SODHIP_ERR_UNSUPPORTED, "porder %d not supported (2..4)", porder);
    }
#undef SODHIP_LPS_CASE
    SODHIP_TRY_HIP(hipGetLastError());
    return SODHIP_OK;
}

template int rhs_fused_elements<double>(sodhip_ctx, int, const MeshCache *, const double *,
                                        const double *, const double *, const int *,
                                        const double *, const double *, const double *,
                                        const double *, double, double, double, double, double,
                                        const double *, double, double, double, double *);
template int rhs_fused_elements<float>(sodhip_ctx, int, const MeshCache *, const float *,
                                       const float *, const float *, const int *, const double *,
                                       const double *, const double *, const float *, double,
                                       double, double, double, double, const double *, double,
                                       double, double, float *);

template <int P, typename T, GradOp OP>
static void launch_grad_p(sodhip_ctx ctx, RhsArgs<T> A, const T *f = nullptr, const T *eta = nullptr)
{
    const UnitShape us = unit_shape<P, T>(ctx, A.nelem);
    A.run = us.run;
    A.wide = us.wide;
    A.geo16 = ((uintptr_t)A.He % 16 == 0) && ((uintptr_t)A.gpvol % 16 == 0);
    k_grad<P, T, OP><<<us.grid, EP<P, T>::NTB, 0, ctx->stream>>>(A, f, eta);
}

template <typename T>
static int scalar_convec(sodhip_ctx ctx, int porder, int nelem, int npoin, const int *connec,
                         const T *He, const T *gpvol, const T *dl, const int *inv, const int *gI,
                         const int *gJ, const int *gK, const T *q, const T *eta, const T *u,
                         T *Rconvec, int initialize, T fact, const EntropyTail *tail = nullptr)
{
    int rc = check_common<T>(ctx, porder, nelem, npoin, connec);
    if (rc) return rc;
    SODHIP_REQUIRE(He && gpvol && dl && inv && gI && gJ && gK && eta && u && (Rconvec || tail),
                   "null array argument");
    SODHIP_TRY_HIP(hipSetDevice(ctx->device));
    MeshCache *m = nullptr;
    if ((rc = get_mesh(ctx, porder, nelem, npoin, connec, &m))) return rc;
    const size_t EN = (size_t)nelem * nnode_of(porder);
    if ((rc = ensure_buf(ctx->scratch, EN * sizeof(T)))) return rc;
    RhsArgs<T> A{};
    A.nelem = nelem;
    A.npoin = npoin;
    A.connecT = m->connecT;
    A.perm = m->perm;
    A.He = He;
    A.gpvol = gpvol;
    A.dl = dl;
    A.inv = inv;
    A.u = u;
    A.out = (T *)ctx->scratch.ptr;
    int tok = prof_begin(ctx, 3);
#define SODHIP_SC(PP)                                              \
    if (q)                                                         \
        launch_grad_p<PP, T, GradOp::SFLUX>(ctx, A, q, eta);       \
    else                                                           \
        launch_grad_p<PP, T, GradOp::SFUSED>(ctx, A, q, eta);
    switch (porder) {
    case 2: SODHIP_SC(2) break;
    case 3: SODHIP_SC(3) break;
    case 4: SODHIP_SC(4) break;
    }
#undef SODHIP_SC
    prof_end(ctx, tok);
    SODHIP_TRY_HIP(hipGetLastError());
    if (tail) {
        if constexpr (std::is_same<T, double>::value) {
            if ((rc = get_working(ctx, m, tail->npoin_w, tail->lpoin_w))) return rc;
            const int bs = 256;
            const int grid = ((tail->npoin_w + bs - 1) / bs + 7) / 8 * 8;
            tok = prof_begin(ctx, 3);
            if (tail->npoin_w > 0)
                k_gather_entropy<<<grid, bs, 0, ctx->stream>>>(npoin, m->wrow, m->wsrc, A.out,
                                                               *tail, fact);
            prof_end(ctx, tok);
            SODHIP_TRY_HIP(hipGetLastError());
            return SODHIP_OK;
        }
        return set_error(SODHIP_ERR_UNSUPPORTED, "entropy residual in FP64 only");
    }
    return launch_gather<T, T>(ctx, m, A.out, 1, Rconvec, nullptr, nullptr, nullptr, nullptr,
                               initialize, fact);
}

// eval_divergence / compute_vorticity / both in one element pass
template <typename T>
static int div_curl(sodhip_ctx ctx, int porder, int nelem, int npoin, int npoin_w,
                    const int *connec, const int *lpoin_w, const int *lelpn, const T *He,
                    const T *gpvol, const T *dl, const int *inv, const int *gI, const int *gJ,
                    const int *gK, const T *u, T *divU, T *curlU)
{
    int rc = check_common<T>(ctx, porder, nelem, npoin, connec);
    if (rc) return rc;
    SODHIP_REQUIRE(He && dl && inv && gI && gJ && gK && u && (divU || curlU),
                   "null array argument");
    SODHIP_REQUIRE(!divU || gpvol, "null gpvol");
    SODHIP_REQUIRE(!curlU || !lelpn || (lpoin_w && npoin_w > 0 && npoin_w <= npoin),
                   "null lpoin_w or invalid npoin_w");
    SODHIP_TRY_HIP(hipSetDevice(ctx->device));
    MeshCache *m = nullptr;
    if ((rc = get_mesh(ctx, porder, nelem, npoin, connec, &m))) return rc;
    const int nf = (divU ? 1 : 0) + (curlU ? 3 : 0);
    const size_t EN = (size_t)nelem * nnode_of(porder);
    if ((rc = ensure_buf(ctx->scratch, nf * EN * sizeof(T)))) return rc;
    RhsArgs<T> A{};
    A.nelem = nelem;
    A.npoin = npoin;
    A.connecT = m->connecT;
    A.perm = m->perm;
    A.He = He;
    A.gpvol = gpvol; // not read where only the vorticity is asked for
    A.dl = dl;
    A.inv = inv;
    A.u = u;
    A.out = (T *)ctx->scratch.ptr;
    int tok = prof_begin(ctx, 3);
#define SODHIP_DC_P(PP)                                                       \
    if (divU && curlU) launch_grad_p<PP, T, GradOp::DIVCURL>(ctx, A);         \
    else if (divU) launch_grad_p<PP, T, GradOp::DIV>(ctx, A);                 \
    else launch_grad_p<PP, T, GradOp::CURL>(ctx, A);
    switch (porder) {
    case 2: SODHIP_DC_P(2) break;
    case 3: SODHIP_DC_P(3) break;
    case 4: SODHIP_DC_P(4) break;
    }
#undef SODHIP_DC_P
    SODHIP_TRY_HIP(hipGetLastError());
    T *c0 = curlU, *c1 = curlU ? curlU + npoin : nullptr, *c2 = curlU ? curlU + 2 * (size_t)npoin : nullptr;
    if (divU && curlU)
        rc = launch_gather<T, T>(ctx, m, A.out, 4, divU, c0, c1, c2, nullptr, 1, T(1));
    else if (divU)
        rc = launch_gather<T, T>(ctx, m, A.out, 1, divU, nullptr, nullptr, nullptr, nullptr, 1,
                                 T(1));
    else
        rc = launch_gather<T, T>(ctx, m, A.out, 3, c0, c1, c2, nullptr, nullptr, 1, T(1));
    if (rc == SODHIP_OK && curlU && lelpn) {
        k_per_elem_count<T><<<(npoin_w + 255) / 256, 256, 0, ctx->stream>>>(npoin, npoin_w, lpoin_w,
                                                                           lelpn, curlU);
        SODHIP_TRY_HIP(hipGetLastError());
    }
    prof_end(ctx, tok);
    return rc;
}

} // namespace sodhip

using namespace sodhip;

extern "C" int sodhip_full_convec_ijk_f64(sodhip_ctx ctx, int porder, int nelem, int npoin,
                                          const int *connec, const double *He,
                                          const double *gpvol, const double *dlxigp_ip,
                                          const int *invAtoIJK, const int *gmshAtoI,
                                          const int *gmshAtoJ, const int *gmshAtoK,
                                          const double *u, const double *q, const double *rho,
                                          const double *pr, const double *E, double *Rmass,
                                          double *Rmom, double *Rener, int initialize,
                                          double fact)
{
    return full_convec<double>(ctx, porder, nelem, npoin, connec, He, gpvol, dlxigp_ip, invAtoIJK,
                               gmshAtoI, gmshAtoJ, gmshAtoK, u, q, rho, pr, E, Rmass, Rmom, Rener,
                               initialize, fact);
}

extern "C" int sodhip_full_convec_ijk_f32(sodhip_ctx ctx, int porder, int nelem, int npoin,
                                          const int *connec, const float *He, const float *gpvol,
                                          const float *dlxigp_ip, const int *invAtoIJK,
                                          const int *gmshAtoI, const int *gmshAtoJ,
                                          const int *gmshAtoK, const float *u, const float *q,
                                          const float *rho, const float *pr, const float *E,
                                          float *Rmass, float *Rmom, float *Rener, int initialize,
                                          float fact)
{
    return full_convec<float>(ctx, porder, nelem, npoin, connec, He, gpvol, dlxigp_ip, invAtoIJK,
                              gmshAtoI, gmshAtoJ, gmshAtoK, u, q, rho, pr, E, Rmass, Rmom, Rener,
                              initialize, fact);
}

extern "C" int sodhip_full_diffusion_ijk_f64(
    sodhip_ctx ctx, int porder, int nelem, int npoin, const int *connec, const double *He,
    const double *gpvol, const double *dlxigp_ip, const int *invAtoIJK, const int *gmshAtoI,
    const int *gmshAtoJ, const int *gmshAtoK, double Cp, double Pr, const double *rho_n,
    const double *rho, const double *u, const double *Tem, const double *mu_fluid,
    const double *mu_e, const double *mu_sgs, double c_rho, double c_ener, double *Rmass,
    double *Rmom, double *Rener, int initialize, double fact)
{
    return full_diffusion<double>(ctx, porder, nelem, npoin, connec, He, gpvol, dlxigp_ip,
                                  invAtoIJK, gmshAtoI, gmshAtoJ, gmshAtoK, Cp, Pr, rho_n, rho, u,
                                  Tem, mu_fluid, mu_e, mu_sgs, c_rho, c_ener, Rmass, Rmom, Rener,
                                  initialize, fact);
}

extern "C" int sodhip_full_diffusion_ijk_f32(
    sodhip_ctx ctx, int porder, int nelem, int npoin, const int *connec, const float *He,
    const float *gpvol, const float *dlxigp_ip, const int *invAtoIJK, const int *gmshAtoI,
    const int *gmshAtoJ, const int *gmshAtoK, float Cp, float Pr, const float *rho_n,
    const float *rho, const float *u, const float *Tem, const float *mu_fluid, const float *mu_e,
    const float *mu_sgs, float c_rho, float c_ener, float *Rmass, float *Rmom, float *Rener,
    int initialize, float fact)
{
    return full_diffusion<float>(ctx, porder, nelem, npoin, connec, He, gpvol, dlxigp_ip,
                                 invAtoIJK, gmshAtoI, gmshAtoJ, gmshAtoK, Cp, Pr, rho_n, rho, u,
                                 Tem, mu_fluid, mu_e, mu_sgs, c_rho, c_ener, Rmass, Rmom, Rener,
                                 initialize, fact);
}

extern "C" int sodhip_generic_scalar_convec_ijk_f64(
    sodhip_ctx ctx, int porder, int nelem, int npoin, const int *connec, const double *He,
    const double *gpvol, const double *dlxigp_ip, const int *invAtoIJK, const int *gmshAtoI,
    const int *gmshAtoJ, const int *gmshAtoK, const double *q, const double *eta,
    const double *u, double *Rconvec, int initialize, double fact)
{
    return scalar_convec<double>(ctx, porder, nelem, npoin, connec, He, gpvol, dlxigp_ip,
                                 invAtoIJK, gmshAtoI, gmshAtoJ, gmshAtoK, q, eta, u, Rconvec,
                                 initialize, fact);
}

extern "C" int sodhip_generic_scalar_convec_ijk_f32(
    sodhip_ctx ctx, int porder, int nelem, int npoin, const int *connec, const float *He,
    const float *gpvol, const float *dlxigp_ip, const int *invAtoIJK, const int *gmshAtoI,
    const int *gmshAtoJ, const int *gmshAtoK, const float *q, const float *eta, const float *u,
    float *Rconvec, int initialize, float fact)
{
    return scalar_convec<float>(ctx, porder, nelem, npoin, connec, He, gpvol, dlxigp_ip,
                                invAtoIJK, gmshAtoI, gmshAtoJ, gmshAtoK, q, eta, u, Rconvec,
                                initialize, fact);
}

extern "C" int sodhip_entropy_convec_residual_f64(
    sodhip_ctx ctx, int porder, int nelem, int npoin, int npoin_w, const int *connec,
    const int *lpoin_w, const double *He, const double *gpvol, const double *dlxigp_ip,
    const int *invAtoIJK, const int *gmshAtoI, const int *gmshAtoJ, const int *gmshAtoK,
    const double *u, const double *eta, const double *invMl, double factor_comp, double dt,
    double *Reta, double *auxReta)
{
    SODHIP_REQUIRE(lpoin_w && eta && invMl && Reta && auxReta, "null array argument");
    SODHIP_REQUIRE(npoin_w >= 0 && npoin_w <= npoin, "npoin_w outside 0..npoin");
    EntropyTail t{npoin_w, lpoin_w, invMl, eta, factor_comp, dt, Reta, auxReta};
    return scalar_convec<double>(ctx, porder, nelem, npoin, connec, He, gpvol, dlxigp_ip,
                                 invAtoIJK, gmshAtoI, gmshAtoJ, gmshAtoK, nullptr, eta, u,
                                 nullptr, 1, 1.0, &t);
}

extern "C" int sodhip_eval_divergence_f64(sodhip_ctx ctx, int porder, int nelem, int npoin,
                                          const int *connec, const double *He,
                                          const double *gpvol, const double *dlxigp_ip,
                                          const int *invAtoIJK, const int *gmshAtoI,
                                          const int *gmshAtoJ, const int *gmshAtoK,
                                          const double *u, double *divU)
{
    return div_curl<double>(ctx, porder, nelem, npoin, 0, connec, nullptr, nullptr, He, gpvol,
                            dlxigp_ip, invAtoIJK, gmshAtoI, gmshAtoJ, gmshAtoK, u, divU, nullptr);
}

extern "C" int sodhip_compute_vorticity_f64(sodhip_ctx ctx, int porder, int nelem, int npoin,
                                            int npoin_w, const int *lpoin_w, const int *connec,
                                            const int *lelpn, const double *He,
                                            const double *dlxigp_ip, const int *invAtoIJK,
                                            const int *gmshAtoI, const int *gmshAtoJ,
                                            const int *gmshAtoK, const double *u, double *curlU)
{
    return div_curl<double>(ctx, porder, nelem, npoin, npoin_w, connec, lpoin_w, lelpn, He,
                            nullptr, dlxigp_ip, invAtoIJK, gmshAtoI, gmshAtoJ, gmshAtoK, u,
                            nullptr, curlU);
}

extern "C" int sodhip_div_curl_f64(sodhip_ctx ctx, int porder, int nelem, int npoin, int npoin_w,
                                   const int *lpoin_w, const int *connec, const int *lelpn,
                                   const double *He, const double *gpvol,
                                   const double *dlxigp_ip, const int *invAtoIJK,
                                   const int *gmshAtoI, const int *gmshAtoJ, const int *gmshAtoK,
                                   const double *u, double *divU, double *curlU)
{
    SODHIP_REQUIRE(divU && curlU, "null output");
    return div_curl<double>(ctx, porder, nelem, npoin, npoin_w, connec, lpoin_w, lelpn, He, gpvol,
                            dlxigp_ip, invAtoIJK, gmshAtoI, gmshAtoJ, gmshAtoK, u, divU, curlU);
}
