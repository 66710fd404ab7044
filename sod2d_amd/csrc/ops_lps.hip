// ops_lps.hip -- local-projection stabilisation of the viscous operator
// (elem_stab.f90): the element time scale comp_tau, the lumped L2 projections
// of the gradients full_proj_ijk, and the stabilised viscous operator
// full_diff_stab_ijk, with their drop-in C-ABI entry points (FP64).
//
// The element kernels of the projections and of the stabilised operator are forms
// of k_rhs (ops_element.hip); their records are gathered per node in the reference's
// (element, node) order by the kernels here (deterministic, no atomics).
#include "common.hpp"
#include "device.hpp"
#include "element.hpp"

namespace sodhip {

// comp_tau (elem_stab.f90:589-616): tau_e = max over the element's nodes of
// h (fact_c c + |u|), h = helem_k (c_species_stab / p), over tiles of 16 elements
// (device.hpp), all loads of an i-line issued together (fmax is exact).
template <int KA>
__global__ __launch_bounds__(256) void k_comp_tau(int nelem, int nnode, int porder,
                                                  const int *__restrict__ connec,
                                                  const int *__restrict__ perm,
                                                  const double *__restrict__ csound,
                                                  const double *__restrict__ u, int npoin,
                                                  const double *__restrict__ helem_k,
                                                  double c_species_stab, double fact_c,
                                                  double *__restrict__ tau)
{
    __shared__ double sh[64];
    __shared__ int alex[125];
    build_alex(perm, nnode, alex);
    constexpr int nl = KA * KA;
    const TileRange tr = tile_range(nelem);
    for (int t = tr.first; t < tr.end; t += tr.stride) {
        const int el = t * kTile + (threadIdx.x & 15), e = min(el, nelem - 1);
        const double h = helem_k[e] * (c_species_stab / (double)porder);
        double taul = 0.0;
        for (int l = threadIdx.x >> 4; l < nl; l += 16) {
            int n[KA];
#pragma unroll
            for (int j = 0; j < KA; ++j)
                n[j] = connec[e + (size_t)nelem * alex[l * KA + j]] - 1;
            double u0[KA], u1[KA], u2[KA], cs[KA];
#pragma unroll
            for (int j = 0; j < KA; ++j) {
                u0[j] = u[n[j]];
                u1[j] = u[n[j] + (size_t)npoin];
                u2[j] = u[n[j] + 2 * (size_t)npoin];
                cs[j] = csound[n[j]];
            }
#pragma unroll
            for (int j = 0; j < KA; ++j) {
                const double aux1 = fact_c * cs[j] + sqrt(u0[j] * u0[j] + u1[j] * u1[j] + u2[j] * u2[j]);
                taul = fmax(taul, h * aux1);
            }
        }
        taul = tile_max(taul, sh);
        if (threadIdx.x < kTile && el < nelem) tau[e] = taul;
    }
}

// Node-ordered assemblies.  Node n's slots row[n]..row[n+1]-1 are taken four
// at a time with every record load issued before the additions, which stay in
// slot order: R_f(n) = (init ? 0 : R_f(n)) + sum_j fact * rec_j[f].  Blocks are
// mapped XCD-aware (the nodes of one XCD are one contiguous range).
__device__ __forceinline__ int xcd_node(int nthr)
{
    const int per = gridDim.x >> 3; // grid is a multiple of 8
    const int blk = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    const int n = blk * blockDim.x + threadIdx.x;
    return n < nthr ? n : -1;
}

struct Rec5Out {
    double *R[5];
};
__global__ __launch_bounds__(256) void k_gather5(int npoin, const int *__restrict__ row,
                                                 const int *__restrict__ src,
                                                 const double *__restrict__ scr, Rec5Out out,
                                                 int init, double fact)
{
    const int n = xcd_node(npoin);
    if (n < 0) return;
    const int j0 = row[n], j1 = row[n + 1];
    double acc[5];
#pragma unroll
    for (int f = 0; f < 5; ++f) acc[f] = init ? 0.0 : out.R[f][n];
    for (int j = j0; j < j1; j += 4) {
        int sj[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) sj[u] = j + u < j1 ? src[j + u] : -1;
        double v[4][5];
#pragma unroll
        for (int u = 0; u < 4; ++u) load_rec5(scr, max(sj[u], 0), v[u]); // absent: not added
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (sj[u] >= 0) {
#pragma unroll
                for (int f = 0; f < 5; ++f) acc[f] += fact * v[u][f];
            }
    }
#pragma unroll
    for (int f = 0; f < 5; ++f) out.R[f][n] = acc[f];
}

// full_proj_ijk's assembly and lumped solve: the 12-value records summed per
// node (the projections start from zero, elem_stab.f90:466-472), scaled by
// invMl on the working nodes (lumped_solver_vect_opt, :576-581), and written
// as ProjMX/MY/MZ (rows of the symmetric tensor), ProjMass, ProjEner.
struct ProjOut {
    double *MX, *MY, *MZ, *Mass, *Ener; // the reference's arrays, or all NULL
    double *prj;                        // one record of kProjRec values per node, or NULL
};
__global__ __launch_bounds__(256) void k_gather_proj(int npoin, const int *__restrict__ row,
                                                     const int *__restrict__ src,
                                                     const double *__restrict__ scr,
                                                     const unsigned char *__restrict__ wflag,
                                                     const double *__restrict__ invMl,
                                                     ProjOut out)
{
    const int n = xcd_node(npoin);
    if (n < 0) return;
    const int j0 = row[n], j1 = row[n + 1];
    double acc[12];
#pragma unroll
    for (int f = 0; f < 12; ++f) acc[f] = 0.0;
    // two slots per step; the loads of an absent slot read record 0 (always
    // present) unconditionally, which is cheaper than masking each load, and
    // are not added
    for (int j = j0; j < j1; j += 2) {
        int sj[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) sj[u] = j + u < j1 ? src[j + u] : -1;
        double2 v[2][6];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const double2 *r = (const double2 *)(scr + 12 * (size_t)max(sj[u], 0));
#pragma unroll
            for (int q = 0; q < 6; ++q) v[u][q] = r[q];
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (sj[u] >= 0) {
#pragma unroll
                for (int q = 0; q < 6; ++q) {
                    acc[2 * q] += v[u][q].x;
                    acc[2 * q + 1] += v[u][q].y;
                }
            }
    }
    if (wflag[n]) {
        const double m = invMl[n];
#pragma unroll
        for (int f = 0; f < 12; ++f) acc[f] *= m;
    }
    if (out.MX) {
        const size_t n1 = n + (size_t)npoin, n2 = n + 2 * (size_t)npoin;
        out.MX[n] = acc[0];
        out.MX[n1] = acc[1];
        out.MX[n2] = acc[2];
        out.MY[n] = acc[1];
        out.MY[n1] = acc[3];
        out.MY[n2] = acc[4];
        out.MZ[n] = acc[2];
        out.MZ[n1] = acc[4];
        out.MZ[n2] = acc[5];
        out.Mass[n] = acc[6];
        out.Mass[n1] = acc[7];
        out.Mass[n2] = acc[8];
        out.Ener[n] = acc[9];
        out.Ener[n1] = acc[10];
        out.Ener[n2] = acc[11];
    }
    if (out.prj) {
        double2 *r = (double2 *)(out.prj + kProjRec * (size_t)n);
#pragma unroll
        for (int q = 0; q < 6; ++q) r[q] = make_double2(acc[2 * q], acc[2 * q + 1]);
    }
}

static int node_grid(int npoin) { return ((npoin + 255) / 256 + 7) / 8 * 8; }

static int lps_common(sodhip_ctx ctx, int porder, int nelem, int npoin, const int *connec,
                      const double *He, const double *gpvol, const double *dl, const int *inv,
                      const int *gI, const int *gJ, const int *gK, MeshCache **m)
{
    SODHIP_REQUIRE(ctx, "null context");
    SODHIP_REQUIRE(porder >= 2 && porder <= kMaxP, "porder %d not supported (2..4)", porder);
    SODHIP_REQUIRE(nelem > 0 && npoin > 0 && connec, "invalid mesh arguments");
    SODHIP_REQUIRE(He && gpvol && dl && inv && gI && gJ && gK, "null array argument");
    SODHIP_TRY_HIP(hipSetDevice(ctx->device));
    return get_mesh(ctx, porder, nelem, npoin, connec, m);
}

// full_proj_ijk into the caller's projections, records through out (12 x EN)
static int proj_run(sodhip_ctx ctx, int porder, const MeshCache *m, LpsArgs A,
                    const double *invMl, double *ProjMass, double *ProjEner, double *ProjMX,
                    double *ProjMY, double *ProjMZ, double *prj = nullptr)
{
    int tok = prof_begin(ctx, 4);
    const int rc = lps_elements(ctx, porder, m, A, LpsKernel::proj);
    if (rc) return rc;
    k_gather_proj<<<node_grid(m->npoin), 256, 0, ctx->stream>>>(
        m->npoin, m->row, m->src, A.out, m->wflag, invMl,
        ProjOut{ProjMX, ProjMY, ProjMZ, ProjMass, ProjEner, prj});
    SODHIP_TRY_HIP(hipGetLastError());
    prof_end(ctx, tok);
    return SODHIP_OK;
}

} // namespace sodhip

using namespace sodhip;

extern "C" int sodhip_comp_tau_f64(sodhip_ctx ctx, int porder, int nelem, int npoin,
                                   const int *connec, const double *csound, const double *u,
                                   const double *helem_k, double c_species_stab,
                                   int flag_drop_c_in_envit, double *tau)
{
    SODHIP_REQUIRE(ctx, "null context");
    SODHIP_REQUIRE(porder >= 2 && porder <= kMaxP, "porder %d not supported (2..4)", porder);
    SODHIP_REQUIRE(nelem > 0 && npoin > 0, "invalid mesh arguments");
    SODHIP_REQUIRE(connec && csound && u && helem_k && tau, "null array argument");
    SODHIP_TRY_HIP(hipSetDevice(ctx->device));
    const int nn = nnode_of(porder);
    MeshCache *m = nullptr;
    int rc = get_mesh(ctx, porder, nelem, npoin, connec, &m);
    if (rc) return rc;
    const int grid = tile_grid(nelem, ctx->num_cu);
#define SODHIP_TAU(KA)                                                                     \
    k_comp_tau<KA><<<grid, 256, 0, ctx->stream>>>( \
        nelem, nn, porder, connec, m->perm, csound, u, npoin, helem_k, c_species_stab, \
        flag_drop_c_in_envit ? 0.0 : 1.0, tau)
    SODHIP_BY_LINE(porder, SODHIP_TAU);
#undef SODHIP_TAU
    SODHIP_TRY_HIP(hipGetLastError());
    return SODHIP_OK;
}

extern "C" int sodhip_full_proj_ijk_f64(sodhip_ctx ctx, int porder, int nelem, int npoin,
                                        int npoin_w, const int *connec, const int *lpoin_w,
                                        const double *He, const double *gpvol,
                                        const double *dlxigp_ip, const int *invAtoIJK,
                                        const int *gmshAtoI, const int *gmshAtoJ,
                                        const int *gmshAtoK, const double *rho, const double *u,
                                        const double *Tem, const double *invMl,
                                        double *ProjMass, double *ProjEner, double *ProjMX,
                                        double *ProjMY, double *ProjMZ)
{
    MeshCache *m = nullptr;
    int rc = lps_common(ctx, porder, nelem, npoin, connec, He, gpvol, dlxigp_ip, invAtoIJK,
                        gmshAtoI, gmshAtoJ, gmshAtoK, &m);
    if (rc) return rc;
    SODHIP_REQUIRE(rho && u && Tem && invMl && lpoin_w && ProjMass && ProjEner && ProjMX &&
                       ProjMY && ProjMZ,
                   "null array argument");
    SODHIP_REQUIRE(npoin_w > 0 && npoin_w <= npoin, "invalid npoin_w");
    const size_t EN = (size_t)nelem * nnode_of(porder);
    if ((rc = ensure_buf(ctx->scratch, 12 * EN * sizeof(double)))) return rc;
    if ((rc = get_working(ctx, m, npoin_w, lpoin_w))) return rc;
    LpsArgs A{};
    A.He = He;
    A.gpvol = gpvol;
    A.dl = dlxigp_ip;
    A.inv = invAtoIJK;
    A.rho = rho;
    A.u = u;
    A.Tem = Tem;
    A.out = (double *)ctx->scratch.ptr;
    return proj_run(ctx, porder, m, A, invMl, ProjMass, ProjEner, ProjMX, ProjMY, ProjMZ);
}

extern "C" int sodhip_full_diff_stab_ijk_f64(
    sodhip_ctx ctx, int porder, int nelem, int npoin, const int *connec, const double *He,
    const double *gpvol, const double *dlxigp_ip, const int *invAtoIJK, const int *gmshAtoI,
    const int *gmshAtoJ, const int *gmshAtoK, double Cp, double Pr, const double *rho_n,
    const double *rho, const double *u, const double *Tem, const double *mu_fluid,
    const double *mu_e, const double *mu_sgs, const double *ProjMass, const double *ProjEner,
    const double *ProjMX, const double *ProjMY, const double *ProjMZ, const double *tau_stab,
    double c_rho, double c_ener, double c_lps, double *Rmass, double *Rmom, double *Rener,
    int initialize, double fact)
{
    MeshCache *m = nullptr;
    int rc = lps_common(ctx, porder, nelem, npoin, connec, He, gpvol, dlxigp_ip, invAtoIJK,
                        gmshAtoI, gmshAtoJ, gmshAtoK, &m);
    if (rc) return rc;
    SODHIP_REQUIRE(rho_n && rho && u && Tem && mu_fluid && mu_e && ProjMass && ProjEner &&
                       ProjMX && ProjMY && ProjMZ && tau_stab && Rmass && Rmom && Rener,
                   "null array argument");
    const size_t EN = (size_t)nelem * nnode_of(porder);
    if ((rc = ensure_buf(ctx->scratch, 5 * EN * sizeof(double)))) return rc;
    LpsArgs A{};
    A.He = He;
    A.gpvol = gpvol;
    A.dl = dlxigp_ip;
    A.inv = invAtoIJK;
    A.rho_n = rho_n;
    A.rho = rho;
    A.u = u;
    A.Tem = Tem;
    A.mu_fluid = mu_fluid;
    A.mu_e = mu_e;
    A.mu_sgs = mu_sgs;
    A.pMass = ProjMass;
    A.pEner = ProjEner;
    A.pMX = ProjMX;
    A.pMY = ProjMY;
    A.pMZ = ProjMZ;
    A.tau = tau_stab;
    A.Cp = Cp;
    A.Pr = Pr;
    A.c_rho = c_rho;
    A.c_ener = c_ener;
    A.c_lps = c_lps;
    A.out = (double *)ctx->scratch.ptr;
    int tok = prof_begin(ctx, 0);
    if ((rc = lps_elements(ctx, porder, m, A, LpsKernel::stab))) return rc;
    prof_end(ctx, tok);
    Rec5Out o{{Rmass, Rmom, Rmom + npoin, Rmom + 2 * (size_t)npoin, Rener}};
    tok = prof_begin(ctx, 1);
    k_gather5<<<node_grid(npoin), 256, 0, ctx->stream>>>(npoin, m->row, m->src, A.out, o,
                                                          initialize, fact);
    SODHIP_TRY_HIP(hipGetLastError());
    prof_end(ctx, tok);
    return SODHIP_OK;
}

extern "C" int sodhip_rk_stage_lps_f64(
    sodhip_ctx ctx, int porder, int nelem, int npoin, int npoin_w, const int *connec,
    const int *lpoin_w, const double *He, const double *gpvol, const double *dlxigp_ip,
    const int *invAtoIJK, const int *gmshAtoI, const int *gmshAtoJ, const int *gmshAtoK,
    const double *mu_e, const double *invMl, const double *tau_stab,
    const sodhip_stage_params *prm, double c_lps, double dt, double lam1, double lams,
    double gam, const double *rho1, const double *q1, const double *E1, double *rho, double *q,
    double *E, double *u, double *e_int, double *pr, double *aux_h, double *Tem,
    double *mu_fluid, double *ProjMass, double *ProjEner, double *ProjMX, double *ProjMY,
    double *ProjMZ, double *Rmass, double *Rmom, double *Rener, double gam_next,
    double *rho_next, double *q_next, double *E_next)
{
    SODHIP_REQUIRE(prm, "null argument");
    MeshCache *m = nullptr;
    int rc = lps_common(ctx, porder, nelem, npoin, connec, He, gpvol, dlxigp_ip, invAtoIJK,
                        gmshAtoI, gmshAtoJ, gmshAtoK, &m);
    if (rc) return rc;
    SODHIP_REQUIRE(lpoin_w && npoin_w > 0 && npoin_w <= npoin, "invalid working nodes");
    SODHIP_REQUIRE(mu_e && invMl && tau_stab && rho1 && q1 && E1 && rho && q && E && u &&
                       e_int && pr && aux_h && Tem && mu_fluid,
                   "null array argument");
    SODHIP_REQUIRE(!!ProjMass == !!ProjEner && !!ProjEner == !!ProjMX && !!ProjMX == !!ProjMY &&
                       !!ProjMY == !!ProjMZ,
                   "ProjMass/ProjEner/ProjMX/ProjMY/ProjMZ: all or none");
    SODHIP_REQUIRE(!!Rmass == !!Rmom && !!Rmom == !!Rener, "Rmass/Rmom/Rener: all or none");
    SODHIP_REQUIRE(!!rho_next == !!q_next && !!q_next == !!E_next, "next stage: all or none");
    SODHIP_REQUIRE(!rho_next || (rho_next != rho && q_next != q && E_next != E),
                   "the next stage must not overwrite the new state");
    if ((rc = get_working(ctx, m, npoin_w, lpoin_w))) return rc;
    // updateF's EOS block and Sutherland's law (time_integ_ls.f90:572-599)
    if ((rc = eos_stage_sutherland(ctx, m, prm->gamma_gas, prm->Rgas, prm->mu_factor, rho, q, E, u,
                                   e_int, pr, aux_h, Tem, mu_fluid)))
        return rc;
    const size_t EN = (size_t)nelem * nnode_of(porder);
    // the projection records start on a 256-byte boundary (their gathers read
    // them with 16-byte loads, and 5*EN doubles is odd when EN is)
    const size_t prec_at = (5 * EN + 31) & ~(size_t)31;
    // then the node projection records, on a 256-byte boundary
    const size_t prj_at = (prec_at + 12 * EN + 31) & ~(size_t)31;
    if ((rc = ensure_buf(ctx->scratch, (prj_at + kProjRec * (size_t)npoin) * sizeof(double))))
        return rc;
    double *rec = (double *)ctx->scratch.ptr, *prec = rec + prec_at, *prj = rec + prj_at;
    // the convection and the stabilised viscous operator run in one element kernel
    // after the projections
    LpsArgs A{};
    A.He = He;
    A.gpvol = gpvol;
    A.dl = dlxigp_ip;
    A.inv = invAtoIJK;
    A.rho = rho;
    A.u = u;
    A.Tem = Tem;
    A.cr = rho;
    A.cq = q;
    A.cE = E;
    A.gamma = prm->gamma_gas;
    A.Rgas = prm->Rgas;
    A.mu_factor = prm->mu_factor;
    A.mu_e = mu_e;
    A.prj = prj;
    A.tau = tau_stab;
    A.Cp = prm->Cp;
    A.Pr = prm->Pr;
    A.c_rho = prm->c_rho;
    A.c_ener = prm->c_ener;
    A.c_lps = c_lps;
    // projections (elem_stab.f90:441-586)
    A.out = prec;
    if ((rc = proj_run(ctx, porder, m, A, invMl, ProjMass, ProjEner, ProjMX, ProjMY, ProjMZ,
                       prj)))
        return rc;
    // both operators carry the same fact (-1), applied once by the gather
    A.out = rec;
    int tok = prof_begin(ctx, 0);
    if ((rc = lps_elements(ctx, porder, m, A, LpsKernel::stage))) return rc;
    prof_end(ctx, tok);
    const NextStage nx{1.0, gam_next * dt, rho_next, q_next, E_next};
    return gather_update<double>(ctx, m, npoin, npoin_w, lpoin_w, rec, 5, EN, invMl, prm->fact, dt,
                                 lam1, lams, gam, rho1, q1, E1, rho, q, E, Rmass, Rmom, Rener,
                                 rho_next ? &nx : nullptr);
}
