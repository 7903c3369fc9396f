// hm_diffusive.hip -- kernels and C-ABI of the diffusive flux of the
// four-equation conservative model (node-based SIXTH_ORDER reconstructor,
// DiffusiveFluxReconstructorNode.cpp:32-1738 with
// DiffusiveFluxReconstructorNodeSixthOrder.cpp:65-939; variables and
// diffusivities of FlowModelDiffusiveFluxUtilitiesFourEqnConservative.cpp:
// 764-1821, 1824-2953, 5673-6425).  Every expression keeps the reference's
// tree, so that with uncontracted arithmetic the result is bit-identical.
#include "hm_ctx.hpp"

namespace hm {

namespace {

template <int D>
__device__ __forceinline__ int dext(const DiffPatch& P, int a) {
    return (a < D) ? P.n[a] + 2 * kGd : 1;
}

template <int D>
__device__ __forceinline__ int64_t dcell(const DiffPatch& P, int i, int j, int k) {
    const int e0 = dext<D>(P, 0), e1 = dext<D>(P, 1);
    return (i + kGd) + int64_t(j + ((D > 1) ? kGd : 0)) * e0 + int64_t(k + ((D > 2) ? kGd : 0)) * e0 * e1;
}

template <int D>
__device__ __forceinline__ int64_t dvol(const DiffPatch& P) {
    return int64_t(dext<D>(P, 0)) * dext<D>(P, 1) * dext<D>(P, 2);
}

template <int D>
__device__ __forceinline__ int64_t dq_idx(const DiffPatch& P, int i, int j, int k) {
    const int e0 = P.n[0] + 2 * P.gq[0];
    const int e1 = (D > 1) ? P.n[1] + 2 * P.gq[1] : 1;
    const int gy = (D > 1) ? P.gq[1] : 0, gz = (D > 2) ? P.gq[2] : 0;
    return (i + P.gq[0]) + int64_t(j + gy) * e0 + int64_t(k + gz) * e0 * e1;
}

// Component slots of the derived cell data: only what the node fluxes
// differentiate, and the pressure.  The density is the sum of the caller's
// partial densities, and the enthalpies and the mixture's transport
// coefficients follow from Y_i, p and T where a node uses them.  Bound by memory:
// twelve stored components instead of seven took 1.06 ms on a level of 448
// uneven patches, now 0.73 (5.6 TB/s of arrays read and written; how much of
// it reaches HBM is not counted).
template <int D, int NS>
struct DiffSlots {
    static constexpr int Y = 0, U = NS, T = NS + D, P = NS + D + 1;
};

// Element i of one component.  The diffusive flux takes patches of up to 2^31
// cells, so the byte offset does not fit the 32 bits of ldg.
__device__ __forceinline__ double ldw(const double* base, uint32_t i) {
    typedef __attribute__((address_space(1))) const double gdouble;
    return ((gdouble*)base)[i];
}
__device__ __forceinline__ void stw(double* base, uint32_t i, double v) {
    typedef __attribute__((address_space(1))) double gdouble;
    ((gdouble*)base)[i] = v;
}

// Block numbers are XCD-contiguous in both kernels: the rows that neighbouring
// blocks' stencils share then sit in one L2.
__device__ __forceinline__ uint32_t diff_block() { return xcd_block(blockIdx.x, gridDim.x); }

// Cells of the 6-ghost box: mass fractions, velocity, pressure of the
// four-equation model (FlowModelFourEqnConservative.cpp:5034-5086), temperature
// p / ((gamma - 1) c_v rho) (EquationOfStateIdealGas.cpp:6951).  Quotients
// through quot / div_rn round as the divisions do.
template <int D, int NS, class W>
__global__ __launch_bounds__(kBlock) void k_diff_cells(W w, DParams k) {
    const int64_t gid = int64_t(diff_block()) * kBlock + threadIdx.x;
    const DiffPatch* P;
    int ax;
    int64_t loc;
    if (!w.find(gid, P, ax, loc)) return;
    using S = DiffSlots<D, NS>;
    const int e0 = dext<D>(*P, 0), e1 = dext<D>(*P, 1);
    // 32-bit index arithmetic (a work segment has fewer than 2^31 items).
    const uint32_t r = uint32_t(loc) / uint32_t(e0);
    const int i = int(uint32_t(loc) - r * uint32_t(e0)) - kGd;
    const int j = (D > 1) ? int((D > 2) ? r % uint32_t(e1) : r) - kGd : 0;
    const int kk = (D > 2) ? int(r / uint32_t(e1)) - kGd : 0;
    const uint32_t iq = uint32_t(dq_idx<D>(*P, i, j, kk));
    double q[NS + D + 1];
#pragma unroll
    for (int e = 0; e < NS + D + 1; e++) q[e] = ldw(P->Q[e], iq);
    double rho = double(0);
    double Y[NS];
#pragma unroll
    for (int si = 0; si < NS; si++) rho += q[si];
    const double rrho = rcp_rn(rho);
#pragma unroll
    for (int si = 0; si < NS; si++) Y[si] = quot(q[si], rho, rrho);
    double u[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int b = 0; b < D; b++) u[b] = quot(q[NS + b], rho, rrho);
    double ke;
    if constexpr (D == 1)
        ke = u[0] * u[0];
    else if constexpr (D == 2)
        ke = u[0] * u[0] + u[1] * u[1];
    else
        ke = u[0] * u[0] + u[1] * u[1] + u[2] * u[2];
    const double eps_int = quot(q[NS + D], rho, rrho) - double(1) / double(2) * ke;
    double c_p = double(0), c_v = double(0);
#pragma unroll
    for (int si = 0; si < NS; si++) {
        c_p += Y[si] * k.cp[si];
        c_v += Y[si] * k.cv[si];
    }
    const double gmix = div_rn(c_p, c_v);
    const double p = (gmix - double(1)) * rho * eps_int;
    const double T = div_rn(p, (gmix - double(1)) * c_v * rho);
    const int64_t vol = dvol<D>(*P);
    const uint32_t c = uint32_t(loc);  // the segment numbers the box's cells
    double* out = P->cell;
#pragma unroll
    for (int si = 0; si < NS; si++) stw(out + (S::Y + si) * vol, c, Y[si]);
#pragma unroll
    for (int b = 0; b < D; b++) stw(out + (S::U + b) * vol, c, u[b]);
    stw(out + S::T * vol, c, T);
    stw(out + S::P * vol, c, p);
}

// Node fluxes of axis A at the cell of index c in the 6-ghost box and q in the
// caller's; col[comp * kDTile + m * step] holds component comp (Y, u, T) of the
// cell m along A.  Per equation, the terms of derivative axes b = 0..D-1 in the
// reference's order, each diffusivity * derivative added to a sum that starts
// at zero (DiffusiveFluxReconstructorNode.cpp:920-1070), from sixth-order
// central first derivatives (DiffusiveFluxReconstructorNodeSixthOrder.cpp:
// 77-112).  Species densities p / (R_i T) (EquationOfStateIdealGas.cpp:8357),
// enthalpies gamma_i p / ((gamma_i - 1) rho_i) (:6464), mixture viscosities and
// conductivity sum(x_i w_i) / sum(w_i), w_i = Y_i / sqrt(M_i)
// (EquationOfShearViscosityMixingRulesConstant.cpp:497-528).
template <int D, int NS, int A>
__device__ __forceinline__ void diff_node(const DiffPatch& P, uint32_t c, uint32_t q, const DParams& k,
                                          const double* col, int step, double (&Fn)[NS + D + 1]) {
    using S = DiffSlots<D, NS>;
    const int64_t vol = dvol<D>(P);
    const int64_t st[3] = {1, dext<D>(P, 0), int64_t(dext<D>(P, 0)) * dext<D>(P, 1)};
    const double* cd = P.cell;
    auto at = [&](int comp, int64_t shift) { return ldw(cd + (comp * vol + shift), c); };
    const double a_n = double(3) / double(4);
    const double b_n = -double(3) / double(20);
    const double c_n = double(1) / double(60);
    auto along = [&](int comp, int m) { return col[comp * kDTile + m * step]; };
    auto deriv6 = [&](int comp, int b) {
        if (b == A)
            return (a_n * (along(comp, 1) - along(comp, -1)) + b_n * (along(comp, 2) - along(comp, -2)) +
                    c_n * (along(comp, 3) - along(comp, -3))) *
                   P.dxinv[b];
        return (a_n * (at(comp, st[b]) - at(comp, -st[b])) + b_n * (at(comp, 2 * st[b]) - at(comp, -2 * st[b])) +
                c_n * (at(comp, 3 * st[b]) - at(comp, -3 * st[b]))) *
               P.dxinv[b];
    };
    double rho = double(0);
#pragma unroll
    for (int si = 0; si < NS; si++) rho += ldw(P.Q[si], q);
    const double p = at(S::P, 0), T = along(S::T, 0);
    double Y[NS], h[NS], u[D];
    double mu_n = double(0), mv_n = double(0), ka_n = double(0), w_d = double(0);
#pragma unroll
    for (int si = 0; si < NS; si++) {
        Y[si] = along(S::Y + si, 0);
        const double rho_i = div_rn(p, k.R[si] * T);
        h[si] = div_rn(k.gamma[si] * p, (k.gamma[si] - double(1)) * rho_i);
        const double wgt = Y[si] * k.wfac[si];
        mu_n += k.mu[si] * wgt;
        mv_n += k.mu_v[si] * wgt;
        ka_n += k.kappa[si] * wgt;
        w_d += wgt;
    }
    const double rw = rcp_rn(w_d);
    const double mu = quot(mu_n, w_d, rw), mu_v = quot(mv_n, w_d, rw), kap = quot(ka_n, w_d, rw);
#pragma unroll
    for (int b = 0; b < D; b++) u[b] = along(S::U + b, 0);

    // Derivatives along A of Y_i, u_c, T; along b != A of u_A and u_b.
    double dY[NS], dU[D], dT;
#pragma unroll
    for (int si = 0; si < NS; si++) dY[si] = deriv6(S::Y + si, A);
#pragma unroll
    for (int b = 0; b < D; b++) dU[b] = deriv6(S::U + b, A);
    dT = deriv6(S::T, A);
    double dUa[3] = {0.0, 0.0, 0.0}, dUb[3] = {0.0, 0.0, 0.0};  // d u_A / dx_b, d u_b / dx_b
#pragma unroll
    for (int b = 0; b < D; b++) {
        if (b == A) continue;
        dUa[b] = deriv6(S::U + A, b);
        dUb[b] = deriv6(S::U + b, b);
    }

    // Mass equations: -rho D_si dY_si + sum_j rho Y_si D_sj dY_sj (derivative along A only).
#pragma unroll
    for (int si = 0; si < NS; si++) {
        double acc = double(0);
        acc += -rho * k.D[si] * dY[si];
#pragma unroll
        for (int sj = 0; sj < NS; sj++) acc += rho * Y[si] * k.D[sj] * dY[sj];
        Fn[si] = acc;
    }
    // Momentum equations.
#pragma unroll
    for (int cc = 0; cc < D; cc++) {
        double acc = double(0);
#pragma unroll
        for (int b = 0; b < D; b++) {
            if (b == A) {
                if (cc == A)
                    acc += -(double(4) / double(3) * mu + mu_v) * dU[cc];
                else
                    acc += -mu * dU[cc];
            } else if (cc == A) {
                acc += (double(2) / double(3) * mu - mu_v) * dUb[b];
            } else if (cc == b) {
                acc += -mu * dUa[b];
            }
        }
        Fn[NS + cc] = acc;
    }
    // Energy equation.
    {
        double acc = double(0);
#pragma unroll
        for (int b = 0; b < D; b++) {
            if (b == A) {
#pragma unroll
                for (int cc = 0; cc < D; cc++) {
                    if (cc == A)
                        acc += -u[cc] * (double(4) / double(3) * mu + mu_v) * dU[cc];
                    else
                        acc += -u[cc] * mu * dU[cc];
                }
                acc += -kap * dT;
#pragma unroll
                for (int si = 0; si < NS; si++) {
                    acc += -rho * k.D[si] * h[si] * dY[si];
#pragma unroll
                    for (int sj = 0; sj < NS; sj++) acc += rho * Y[si] * k.D[sj] * h[si] * dY[sj];
                }
            } else if (A < b) {
                acc += -u[b] * mu * dUa[b];
                acc += u[A] * (double(2) / double(3) * mu - mu_v) * dUb[b];
            } else {
                acc += u[A] * (double(2) / double(3) * mu - mu_v) * dUb[b];
                acc += -u[b] * mu * dUa[b];
            }
        }
        Fn[NS + D] = acc;
    }
}

// Diffusive flux of axis A over one tile (dtile_shape): R consecutive cells
// along A of W columns, one per thread, staged in LDS (Y, u, T), so that the
// derivatives along A read LDS.  The threads of the cells 3 from either end form
// node fluxes, which then take the cells' places, and the threads with three
// nodes below and two above the output faces
// (DiffusiveFluxReconstructorNodeSixthOrder.cpp:507-690):
// F_face = 0 + dt (a_r (F_L + F_R) + b_r (F_LL + F_RR) + c_r (F_LLL + F_RRR)).
// Every output face has one such thread.  Bound by the caches' load rate: with
// node fluxes to memory and a second kernel the pair took 2.75 + 1.47 ms on a
// level of 448 uneven patches (Navier-Stokes, 6-cell halos) and moved 13 GB;
// fused with every derivative from memory 3.09 ms, now 2.66.  Blocks of 512 threads keep a
// tile's rows 6 cells wide (62 to 73 cells along the axis) to 39 (one cell), and
// XCD-contiguous blocks the lines at their edges in one L2.
template <int D, int NS, int A>
__device__ __forceinline__ void diff_tile(const DiffPatch& P, uint32_t tile, const DParams& k, double* lds) {
    constexpr int NEQ = NS + D + 1;
    const int nA = P.n[A];
    const int R = P.tile[A][0], W = P.tile[A][1], ntA = P.tile[A][2];
    const uint32_t lane = threadIdx.x;
    const uint32_t tw = tile / uint32_t(ntA), tA = tile - tw * uint32_t(ntA);
    uint32_t r, w;
    tile_place(A, lane, uint32_t(R), uint32_t(W), uint32_t(P.tile[A][3]), r, w);
    const int x = int(tA) * (R - kDTileShared) - 6 + int(r);  // cell along A
    constexpr int U = (A == 0) ? 1 : 0;  // first axis across
    constexpr int V = (A == 2) ? 1 : 2;  // second axis across
    uint32_t cu, tv;
    tile_column(tw * uint32_t(W), w, uint32_t(W), uint32_t(D > U ? P.n[U] : 1), cu, tv);
    const bool in = lane < uint32_t(R * W) && x < nA + 6 && tv < uint32_t(D > V ? P.n[V] : 1);
    int i[3];
    i[A] = x;
    i[U] = int(cu);
    i[V] = int(tv);
    const int step = A == 0 ? 1 : W;  // thread distance of neighbouring rows
    const uint32_t c = uint32_t(dcell<D>(P, i[0], i[1], i[2]));
    const int64_t vol = dvol<D>(P);
    if (in) {
#pragma unroll
        for (int e = 0; e < NEQ; e++) lds[e * kDTile + lane] = ldw(P.cell + e * vol, c);  // Y, u, T
    }
    __syncthreads();
    const bool node = in && int(r) >= 3 && int(r) < R - 3 && x < nA + 3;
    double Fn[NEQ];
    if (node)
        diff_node<D, NS, A>(P, c, uint32_t(dq_idx<D>(P, i[0], i[1], i[2])), k, lds + lane, step, Fn);
    __syncthreads();
    if (node) {
#pragma unroll
        for (int e = 0; e < NEQ; e++) lds[e * kDTile + lane] = Fn[e];
    }
    __syncthreads();
    if (!in || int(r) < 6 || int(r) > R - 6 || x > nA) return;  // face x: nodes x - 3 .. x + 2
    const uint32_t f0 = uint32_t(P.n[0] + (A == 0)), f1 = uint32_t(D > 1 ? P.n[1] + (A == 1) : 1);
    const uint32_t fi = uint32_t(i[0]) + f0 * (uint32_t(i[1]) + f1 * uint32_t(i[2]));
    const int64_t fvol = int64_t(f0) * f1 * (D > 2 ? P.n[2] + (A == 2) : 1);
    const double a_n = double(3) / double(4);
    const double b_n = -double(3) / double(20);
    const double c_n = double(1) / double(60);
    const double a_r = a_n + b_n + c_n;
    const double b_r = b_n + c_n;
    const double c_r = c_n;
    double* out = P.F[A];
    const double dt = k.dtp ? *k.dtp : k.dt;
#pragma unroll
    for (int e = 0; e < NEQ; e++) {
        auto f = [&](int m) { return lds[e * kDTile + int(lane) + m * step]; };
        double acc = double(0);
        acc += dt * (a_r * (f(-1) + f(0)) + b_r * (f(-2) + f(1)) + c_r * (f(-3) + f(2)));
        stw(out + e * fvol, fi, acc);
    }
}

template <int D, int NS, class W>
__global__ __launch_bounds__(kDTile) void k_diff_flux(W w, DParams k) {
    __shared__ double lds[(NS + D + 1) * kDTile];
    const DiffPatch* P;
    int A;
    uint32_t tile;
    if (!find_block<kDTile>(w, diff_block(), P, A, tile)) return;  // whole blocks
    if (A == 0) {
        diff_tile<D, NS, 0>(*P, tile, k, lds);
    } else if constexpr (D > 1) {
        if (A == 1) {
            diff_tile<D, NS, 1>(*P, tile, k, lds);
        } else if constexpr (D > 2) {
            diff_tile<D, NS, 2>(*P, tile, k, lds);
        }
    }
}

template <int D, int NS, class W>
hipError_t launch_dn(const DPlan<W>& plan, const DParams& k, hipStream_t s) {
    const unsigned cells = unsigned((plan.items[0] + kBlock - 1) / kBlock), tiles = unsigned(plan.items[1] / kDTile);
    if (cells) hipLaunchKernelGGL((k_diff_cells<D, NS, W>), dim3(cells), dim3(kBlock), 0, s, plan.work[0], k);
    if (tiles) hipLaunchKernelGGL((k_diff_flux<D, NS, W>), dim3(tiles), dim3(kDTile), 0, s, plan.work[1], k);
    return hipGetLastError();
}

template <int D, class W>
hipError_t launch_d(const DPlan<W>& plan, const DParams& k, hipStream_t s) {
    switch (k.num_species) {
        case 1: return launch_dn<D, 1, W>(plan, k, s);
        case 2: return launch_dn<D, 2, W>(plan, k, s);
        case 3: return launch_dn<D, 3, W>(plan, k, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

template <class W>
hipError_t launch_diffusive_four(int dim, const DPlan<W>& plan, const DParams& k, hipStream_t s) {
    switch (dim) {
        case 1: return launch_d<1, W>(plan, k, s);
        case 2: return launch_d<2, W>(plan, k, s);
        case 3: return launch_d<3, W>(plan, k, s);
        default: return hipErrorInvalidValue;
    }
}

template hipError_t launch_diffusive_four<SegSingleT<DiffPatch>>(int, const DPlan<SegSingleT<DiffPatch>>&,
                                                                 const DParams&, hipStream_t);
template hipError_t launch_diffusive_four<SegTableT<DiffPatch>>(int, const DPlan<SegTableT<DiffPatch>>&,
                                                                const DParams&, hipStream_t);

}  // namespace hm

extern "C" {

int hm_set_diffusive_transport(hm_ctx* ctx, const hm_transport* tr) {
    if (!ctx || !ctx->rec) return HM_ERR_INVALID_ARGUMENT;
    if (!tr) return ctx->rec->fail(HM_ERR_INVALID_ARGUMENT, "NULL transport properties");
    const hm_config& c = ctx->rec->config();
    if (c.model != HM_MODEL_FOUR_EQN_CONSERVATIVE)
        return ctx->rec->fail(HM_ERR_UNSUPPORTED, "the diffusive flux is built for the four-equation model");
    for (int i = 0; i < c.num_species; i++) {
        if (!(tr->species_M[i] > 0.0)) return ctx->rec->fail(HM_ERR_INVALID_ARGUMENT, "species_M must be positive");
        if (!(tr->species_mu[i] >= 0.0) || !(tr->species_mu_v[i] >= 0.0) || !(tr->species_kappa[i] >= 0.0) ||
            !(tr->species_D[i] >= 0.0))
            return ctx->rec->fail(HM_ERR_INVALID_ARGUMENT, "transport coefficients must be non-negative");
    }
    if (ctx->levels > 0)
        return ctx->rec->fail(HM_ERR_INVALID_ARGUMENT,
                              "set the transport properties before creating levels on this context");
    if (int st = ctx->rec->selectDevice()) return st;
    ctx->diff.reset();
    ctx->diff.reset(new (std::nothrow) hm::DiffusiveFluxReconstructorGPU(*ctx->rec, *tr));
    if (!ctx->diff) return ctx->rec->fail(HM_ERR_OUT_OF_MEMORY, "out of host memory");
    return HM_OK;
}

int hm_get_diffusive_num_ghosts(const hm_ctx* ctx, int* num_ghosts) {
    if (!ctx || !ctx->diff || !num_ghosts) return HM_ERR_INVALID_ARGUMENT;
    *num_ghosts = ctx->diff->getDiffusiveFluxNumberOfGhostCells();
    return HM_OK;
}

int hm_compute_diffusive_flux_on_patch(hm_ctx* ctx, const hm_patch_view* patch, double time, double dt,
                                       int rk_step, void* stream) {
    if (!ctx || !ctx->rec) return HM_ERR_INVALID_ARGUMENT;
    if (!ctx->diff) return ctx->rec->fail(HM_ERR_INVALID_ARGUMENT, "set the transport properties first");
    if (!patch) return ctx->rec->fail(HM_ERR_INVALID_ARGUMENT, "NULL patch view");
    return ctx->diff->computeDiffusiveFluxOnPatch(*patch, time, dt, rk_step, static_cast<hipStream_t>(stream));
}

int hm_compute_diffusive_flux_on_patches(hm_ctx* ctx, const hm_patch_view* patches, int num_patches, double time,
                                         double dt, int rk_step, void* stream) {
    if (!ctx || !ctx->rec) return HM_ERR_INVALID_ARGUMENT;
    if (!ctx->diff) return ctx->rec->fail(HM_ERR_INVALID_ARGUMENT, "set the transport properties first");
    return ctx->diff->computeDiffusiveFluxOnPatches(patches, num_patches, time, dt, rk_step,
                                                    static_cast<hipStream_t>(stream));
}

}  // extern "C"
