// Per-step physics passes of the ISPH projection step on MI355X.
//
// Structure-of-arrays state; a thread per particle where a pass reads no
// neighbours, else groups of lanes (GROUP; 16 or 32 for the boundary passes; a
// wave for FP64 Neumann sums and heavy MIXED lists), which
// walk the per-particle neighbour list built once by the count==0 search
// (the reference rescans the 5^3 cell window every pass; in its Eulerian mode
// positions never move, ISPH_Calc.cuh:23-63).  Each list entry carries
// precomputed FP64 window/radius flags, so a pass selects exactly the
// reference's neighbour set for that kernel in both precision modes.
// Passes whose search is centred on a ghost node (Neumann inlet mirror,
// periodic copy, outlet copy, MOST deposit) scan the cell window directly.
//
// R is the pair-math type (double: FP64 mode, float: mixed mode).  Sums are
// always accumulated in double.  Differences of positions and velocities are
// taken in double and then rounded to R, so the float path loses no
// significance to cancellation.
#include <string>

#include "flags.h"
#include "sph_internal.h"
#include "sph_math.h"

namespace sph {

// This thread's particle: case descriptor `cd` and index `i` in the case;
// threads past the case's end return.
#define SEG_PARTICLE(sg)                          \
    int first_;                                   \
    const int cid_ = seg_case((sg), first_);      \
    const CaseDesc& cd = (sg).cd[cid_];           \
    const int i = first_ + (int)threadIdx.x;      \
    if (i >= cd.n) return;
// BLANES lanes (lane: this one) per particle of the case's boundary list
// (every p_type but fluid): wall, lid and marker passes, which leave most of
// that list at once, so a wave of its own for each particle mostly waits on
// the loads that lead to its p_type (free slip, 2.13 M canyon: 222 us, with 16
// lanes 131; FP64, 1 M: 380 and 186 us, a thread each 190; 20 k: 13, 14, 65).
constexpr int BLANES = 16;
#define SEG_BOUNDARY(sg) SEG_BOUNDARY_LANES(sg, BLANES)
#define SEG_BOUNDARY_LANES(sg, lanes)                                  \
    int first_;                                                        \
    const int cid_ = seg_case(sg, first_);                             \
    const CaseDesc& cd = sg.cd[cid_];                                  \
    if ((sg).tab == nullptr) first_ *= 64 / (lanes);   /* blocks of blockDim * 64 / lanes */ \
    const int u_ = first_ / 64 + (int)threadIdx.x / (lanes), lane = (int)threadIdx.x % (lanes); \
    if (u_ >= cd.nm_count) return;                                     \
    const int i = cd.nm_list[u_];
// GROUP lanes a particle (g_: the lane in its group)
#define SEG_GROUP(sg)                                     \
    int first_;                                           \
    const int cid_ = seg_case((sg), first_);              \
    const CaseDesc& cd = (sg).cd[cid_];                   \
    const int i = first_ + (int)threadIdx.x / GROUP, g_ = (int)threadIdx.x % GROUP; \
    if (i >= cd.n) return;
// prep, advection and the pressure force: the particles of short lists in the
// pass order; in MIXED the last cd.n_heavy of that order (the heavy lists) are
// left to a wave each (SEG_HEAVY)
#define SEG_GROUP_LIGHT(sg)                               \
    int first_;                                           \
    const int cid_ = seg_case((sg), first_);              \
    const CaseDesc& cd = (sg).cd[cid_];                   \
    const int t_ = first_ + (int)threadIdx.x / GROUP, g_ = (int)threadIdx.x % GROUP; \
    if (t_ >= cd.n - cd.n_heavy) return;                  \
    const int i = cd.porder ? cd.porder[t_] : t_;
#define SEG_HEAVY(sg)                                         \
    int first_;                                               \
    const int cid_ = seg_case((sg), first_);                  \
    const CaseDesc& cd = (sg).cd[cid_];                       \
    const int u_ = (first_ + (int)threadIdx.x) >> 6;          \
    const int lane_ = threadIdx.x & 63;                       \
    if (u_ >= cd.n_heavy) return;                             \
    const int i = cd.porder[cd.n - cd.n_heavy + u_];
// FP64: dynamic LDS of ordered sums, this wave's part
#define ORDERED_LDS(nt, n2)            \
    extern __shared__ double ord_lds_[]; \
    double* const wlds_ = ord_lds_ + (threadIdx.x >> 6) * ord_doubles((nt), (n2));

// Particles of the cells (i0..i1, cj, ck) that lie inside the grid, as one
// range [rg.x, rg.y) of the sorted order; false when the row is outside the
// grid or the clipped x-range is empty.
__device__ __forceinline__ bool row_range(const Grid& g, int i0, int i1, int cj, int ck, int2& rg) {
    const sph_domain& d = g.d;
    if (cj < 0 || cj > d.NJ - 1 || ck < 0 || ck > d.NK - 1) return false;
    i0 = max(i0, 0);
    i1 = min(i1, d.NI - 1);
    if (i0 > i1) return false;
    const int base = d.NI * cj + d.NI * d.NJ * ck;
    rg = make_int2(g.cstart[base + i0], g.cstart[base + i1 + 1]);
    return true;
}

// Bin-cell range that contains every particle within distance r of p
// (binning is monotone in each coordinate; a small margin absorbs the
// double -> float rounding of the bounds).
__device__ __forceinline__ void ball_bins(const sph_domain& d, double px, double py, double pz, double r,
                                          Cell& lo, Cell& hi) {
    const double m = 1e-9 + 1e-6 * r;
    lo = Cell{bin_axis((float)(px - r - m), d.x_min, d.x_max, d.NI), bin_axis((float)(py - r - m), d.y_min, d.y_max, d.NJ),
              bin_axis((float)(pz - r - m), d.z_min, d.z_max, d.NK)};
    hi = Cell{bin_axis((float)(px + r + m), d.x_min, d.x_max, d.NI), bin_axis((float)(py + r + m), d.y_min, d.y_max, d.NJ),
              bin_axis((float)(pz + r + m), d.z_min, d.z_max, d.NK)};
}


// ------------------------------------------------------------------------
// Step start: SP1 <- P1 and SP2 <- P2 for the mutable fields, P3 <- 0
// (ISPH_Calc.cuh:53-63), and KERNEL_set_ncell (functions_NNPS.cuh:943-955).
__global__ void __launch_bounds__(MAX_BLOCK) k_step_begin(Seg sg) {
    SEG_PARTICLE(sg);
    const PView P = cd.P, S = cd.S;
    const P2View P2 = cd.P2, S2 = cd.S2;
    const QView Q = cd.Q;
    if (P.i_type[i] != 3) P.ncell[i] = (int)(1.0 * ceilf(2.0f / (float)(P.h_ref[i] / P.h[i])));
    S.ux[i] = P.ux[i]; S.uy[i] = P.uy[i]; S.uz[i] = P.uz[i]; S.pres[i] = P.pres[i]; S.temp[i] = P.temp[i];
    S.vis_t[i] = P.vis_t[i]; S.k_turb[i] = P.k_turb[i]; S.e_turb[i] = P.e_turb[i]; S.flt_s[i] = P.flt_s[i];
    S.fmx[i] = P.fmx[i]; S.fmy[i] = P.fmy[i]; S.hmz[i] = P.hmz[i];
    S.float1[i] = P.float1[i]; S.float2[i] = P.float2[i]; S.float3[i] = P.float3[i];
    S.fbx[i] = P.fbx[i]; S.fby[i] = P.fby[i]; S.fbz[i] = P.fbz[i];
    S.concentration[i] = P.concentration[i]; S.concn[i] = P.concn[i]; S.enthalpy[i] = P.enthalpy[i];
    S2.rho_ref[i] = P2.rho_ref[i]; S2.SR[i] = P2.SR[i]; S2.x0[i] = P2.x0[i]; S2.y0[i] = P2.y0[i];
    S2.z0[i] = P2.z0[i]; S2.ux0[i] = P2.ux0[i]; S2.uy0[i] = P2.uy0[i]; S2.uz0[i] = P2.uz0[i];
    S2.temp0[i] = P2.temp0[i]; S2.concn0[i] = P2.concn0[i];
    Q.ftotalx[i] = 0.0; Q.ftotaly[i] = 0.0; Q.ftotalz[i] = 0.0; Q.ftotal[i] = 0.0;
    Q.fpx[i] = 0.0; Q.fpy[i] = 0.0; Q.fpz[i] = 0.0; Q.dtemp[i] = 0.0; Q.dconcn[i] = 0.0;
    if (!cd.gc_fresh) {
        Q.inv_xx[i] = 0.0; Q.inv_yy[i] = 0.0; Q.inv_zz[i] = 0.0; Q.inv_xy[i] = 0.0; Q.inv_yz[i] = 0.0; Q.inv_zx[i] = 0.0;
    }
    if (cd.xnew[0]) { cd.xnew[0][i] = P.x[i]; cd.xnew[1][i] = P.y[i]; cd.xnew[2][i] = P.z[i]; }
}

// ALE: the corrector's positions become the state at the end of the step,
// after the boundary passes that still search the step's cells.
__global__ void __launch_bounds__(MAX_BLOCK) k_commit_positions(Seg sg) {
    SEG_PARTICLE(sg);
    if (!cd.xnew[0]) return;
    const PView P = cd.P;
    P.x[i] = cd.xnew[0][i]; P.y[i] = cd.xnew[1][i]; P.z[i] = cd.xnew[2][i];
}

// Snapshot of the fields a copy/mirror pass reads while it writes them.
__global__ void __launch_bounds__(MAX_BLOCK) k_snapshot(Seg sg, int which, int nm_pack) {
    SEG_PARTICLE(sg);
    const PView A = which ? cd.P : cd.S;
    cd.snap[3][i] = A.pres[i];
    if (!nm_pack) {   // (the Neumann pass reads the pressures only)
        cd.snap[0][i] = A.ux[i]; cd.snap[1][i] = A.uy[i]; cd.snap[2][i] = A.uz[i];
        cd.snap[4][i] = A.temp[i];
    }
    if (nm_pack && cd.nm_rec && i < cd.nm_nset) {   // the Neumann pass's records, from the same state
        const int j = cd.nm_set[i];
        const size_t n = (size_t)cd.nm_nset;
        float4* r = (float4*)cd.nm_rec + i;
        r[0] = make_float4((float)A.x[j], (float)A.y[j], (float)A.z[j], (float)A.m[j]);
        r[n] = make_float4((float)A.rho[j], (float)A.ux[j], (float)A.uy[j], (float)A.uz[j]);
        *(double2*)(r + 2 * n) = make_double2(A.pres[j], 0.0);
    }
}

// ------------------------------------------------------------------------
// KERNEL_clc_gradient_correction_3D, functions_KNL.cuh:216-324
// the inverse of the moment matrix of a fluid particle's fluid neighbours
// (the identity where it is singular, and for every other particle)
__device__ __forceinline__ void grad_corr_store(const QView& Q, int i, int ptype_i, double tmpxx, double tmpyy,
                                                double tmpzz, double tmpxy, double tmpyz, double tmpzx) {
    double tmpcmd = tmpxx * (tmpyy * tmpzz - tmpyz * tmpyz);
    tmpcmd -= tmpxy * (tmpxy * tmpzz - tmpyz * tmpzx);
    tmpcmd += tmpzx * (tmpxy * tmpyz - tmpyy * tmpzx);
    if ((fabs(tmpcmd) > 2.2204460492503131e-16) && (ptype_i == 1)) {
        double rtcmd = 1.0 / tmpcmd;
        Q.inv_xx[i] = (tmpyy * tmpzz - tmpyz * tmpyz) * rtcmd;
        Q.inv_xy[i] = (tmpzx * tmpyz - tmpxy * tmpzz) * rtcmd;
        Q.inv_zx[i] = (tmpxy * tmpyz - tmpzx * tmpyy) * rtcmd;
        Q.inv_yy[i] = (tmpxx * tmpzz - tmpzx * tmpzx) * rtcmd;
        Q.inv_yz[i] = (tmpzx * tmpxy - tmpxx * tmpyz) * rtcmd;
        Q.inv_zz[i] = (tmpxx * tmpyy - tmpxy * tmpxy) * rtcmd;
    } else {
        Q.inv_xx[i] = 1.0; Q.inv_xy[i] = 0.0; Q.inv_zx[i] = 0.0;
        Q.inv_yy[i] = 1.0; Q.inv_yz[i] = 0.0; Q.inv_zz[i] = 1.0;
    }
}

constexpr int GC_SUMS = 6;
__global__ void __launch_bounds__(MAX_BLOCK) k_grad_corr(Seg sg) {
    ORDERED_LDS(GC_SUMS, 0);
    SEG_GROUP(sg);
    if (cd.gc_fresh) return;   // unchanged since the last step of this search
    const KConst kc = cd.kc;
    const PView S = cd.S;
    const double hi = S.h[i], tmp_A = calc_tmpA<double>(kc, hi);
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    OrderedSums<GC_SUMS, GROUP> sums(wlds_);   // xx, yy, zz, xy, yz, zx
    const NLRow row = nl_row(cd.nl, i);
    for (int k = g_; k - g_ < row.cnt; k += GROUP) {
        const unsigned e = k < row.cnt ? NB_AT(row, k) : 0u;
        const bool pair = (e & F_B) != 0;
        if (!__any(pair)) continue;
        double v[GC_SUMS] = {};
        if (pair) {
            const int j = e & NB_IDX;
            const double dx = xi - S.x[j], dy = yi - S.y[j], dz = zi - S.z[j];
            const double tdist = sqrt(dx * dx + dy * dy + dz * dz);
            const double tdwij = kernel_dw<double>(kc, tmp_A, hi, tdist);
            const double mj = S.m[j], rhoj = S.rho[j];
            const double mtd = mj * tdwij, rtd = 1.0 / (rhoj * tdist), f = (double)(S.p_type[j] == 1);
            v[0] = -mtd * dx * dx * rtd * f;
            v[1] = -mtd * dy * dy * rtd * f;
            v[2] = -mtd * dz * dz * rtd * f;
            v[3] = -mtd * dy * dx * rtd * f;
            v[4] = -mtd * dy * dz * rtd * f;
            v[5] = -mtd * dx * dz * rtd * f;
        }
        sums.add(v);
    }
    double t[GC_SUMS];
    for (int a = 0; a < GC_SUMS; a++) t[a] = sums.sum(a);
    if (g_ == 0) grad_corr_store(cd.Q, i, S.p_type[i], t[0], t[1], t[2], t[3], t[4], t[5]);
}
// MIXED: GROUP lanes a particle (SEG_GROUP), the pair arithmetic in float,
// the sums in double
__global__ void __launch_bounds__(MAX_BLOCK) k_grad_corr_mixed(Seg sg) {
    SEG_GROUP(sg);
    if (cd.gc_fresh) return;   // unchanged since the last step of this search
    const KConst kc = cd.kc;
    const PView S = cd.S;
    const float hi = (float)S.h[i], tmp_A = calc_tmpA<float>(kc, hi), f = dw_factor<float>(kc, hi);
    const HScale hs(kc, hi);
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    double txx = 0, tyy = 0, tzz = 0, txy = 0, tyz = 0, tzx = 0;
    const NLRow row = nl_row(cd.nl, i);
    for (int k = g_; k < row.cnt; k += GROUP) {
        const unsigned e = NB_AT(row, k);
        if (!(e & F_B)) continue;
        const int j = e & NB_IDX;
        const float dx = (float)(xi - S.x[j]), dy = (float)(yi - S.y[j]), dz = (float)(zi - S.z[j]);
        const Dist d = dist_of(dx * dx + dy * dy + dz * dz);
        const float w = -((float)S.m[j] * kernel_dw_t<float>(kc, tmp_A, f, hs.tR(d.r)));
        const float rtd = 1.0f / ((float)S.rho[j] * d.r), fl = (float)(S.p_type[j] == 1);
        txx += (double)(w * dx * dx * rtd * fl); txy += (double)(w * dy * dx * rtd * fl);
        tyy += (double)(w * dy * dy * rtd * fl); tzx += (double)(w * dx * dz * rtd * fl);
        tyz += (double)(w * dy * dz * rtd * fl); tzz += (double)(w * dz * dz * rtd * fl);
    }
    group_fold<GROUP>(txx); group_fold<GROUP>(tyy); group_fold<GROUP>(tzz);
    group_fold<GROUP>(txy); group_fold<GROUP>(tyz); group_fold<GROUP>(tzx);
    if (g_ != 0) return;
    grad_corr_store(cd.Q, i, S.p_type[i], txx, tyy, tzz, txy, tyz, tzx);
}

// ------------------------------------------------------------------------
// KERNEL_clc_prep3D, functions_PREP.cuh:287-488
// Neighbour records of every particle from the working state (see
// rec_pos): all pairs, or only those that hold velocities and pressures, or
// pressures.
template <int WHICH>
__global__ void __launch_bounds__(BLOCK) k_pack_records(Seg sg) {
    SEG_PARTICLE(sg);
    const PView S = cd.S;
    const size_t n = (size_t)cd.n;   // piece q of particle i: element q * n + i
    if (cd.crec) {   // the gathering passes of this case read the compact records
        if (WHICH == REC_PQ) {
            float4* c = (float4*)cd.crec + i;
            c[0] = make_float4((float)S.x[i], (float)S.y[i], (float)S.z[i], (float)S.m[i]);
            c[n] = make_float4((float)S.rho[i], (float)(S.pres[i] - S.pres0[i]), (float)S.h[i],
                               __int_as_float(S.p_type[i]));
            return;
        }
        float4* c = (float4*)cd.crec_adv + i;
        double2* d = (double2*)(c + 2 * n);
        d[0] = make_double2(S.ux[i], S.uy[i]);
        d[n] = make_double2(S.uz[i], S.pres[i] - S.pres0[i]);
        if (WHICH == REC_VEL_PQ) return;
        const int t = (S.p_type[i] & 0xffff) | (S.i_type[i] << 16) |
                      (cd.ppe.rowof && cd.ppe.rowof[i] >= 0 ? CREC_ROW_BIT : 0);
        if (WHICH == REC_PRE) c[0] = make_float4((float)S.x[i], (float)S.y[i], (float)S.z[i], (float)S.m[i]);
        c[n] = make_float4((float)S.rho[i], (float)S.h[i],
                           (float)(viscosity2(cd.pr, S.p_type[i]) + S.vis_t[i] * S.rho[i]), __int_as_float(t));
        return;
    }
    if (WHICH == REC_PRE) return;
    double2* r = (double2*)cd.rec + i;
    r[2 * n] = make_double2(S.rho[i], S.pres[i] - S.pres0[i]);
    if (WHICH == REC_PQ) return;
    r[3 * n] = make_double2(S.ux[i], S.uy[i]);
    r[4 * n] = make_double2(S.uz[i], S.h[i]);
    if (WHICH == REC_VEL_PQ) return;
    const long long t = (long long)(unsigned)S.p_type[i] | ((long long)S.i_type[i] << 32);
    r[0] = make_double2(S.x[i], S.y[i]);
    r[n] = make_double2(S.z[i], S.m[i]);
    r[5 * n] = make_double2(S.vis_t[i], __longlong_as_double(t));
    r[6 * n] = make_double2(S.temp[i], S.concn[i]);
}

// A particle's strain rate and eddy viscosity from its sums.
__device__ __forceinline__ void prep_store(const CaseDesc& cd, int i, bool les, bool filt, double ki, double nui,
                                           double hi_d, double tmp_flt, double tmp_sigma, double st11, double st12,
                                           double st22, double st23, double st31, double st33) {
    const sph_params& pr = cd.pr;
    const PView S = cd.S;
    const P2View S2 = cd.S2;
    if (les) {
        double tmp_SR = 2 * (st11 * st11 + st22 * st22 + st33 * st33 + 2 * st12 * st12 + 2 * st31 * st31 + 2 * st23 * st23);
        tmp_SR = sqrt(tmp_SR);
        S2.SR[i] = tmp_SR;
        tmp_sigma = 0.3333 * tmp_sigma;
        tmp_sigma = sqrt(tmp_sigma);
        double tmp_cl = tmp_sigma > hi_d ? tmp_sigma : hi_d;
        if (pr.turbulence_model == SPH_SSM) {
            double tvis_t = pr.Cs_sgs * pr.Cs_sgs * tmp_cl * tmp_cl * tmp_SR;
            if (S.buffer_type[i] != 1) S.vis_t[i] = tvis_t;
        } else if (pr.turbulence_model == SPH_DDF) {
            double p = nui * tmp_SR * tmp_SR;
            double b = 0.0;
            double eps = pr.Ce_sgs * ki * sqrt(ki) / tmp_cl;
            double dk = p + b - eps + 0.0;
            ki += dk * cd.dt;
            ki = ki > 1e-4 ? ki : 1e-4;
            double tvis_t = pr.Ck_sgs * tmp_cl * sqrt(ki);
            if (S.buffer_type[i] != 1) { S.vis_t[i] = tvis_t; S.k_turb[i] = ki; S.e_turb[i] = eps; }
        }
    }
    if (cd.count == 0) S2.rho_ref[i] = S.rho[i];
    if (filt) S.flt_s[i] = tmp_flt;
}
constexpr int PREP_SUMS = 8;
__global__ void __launch_bounds__(MAX_BLOCK) k_prep(Seg sg) {
    ORDERED_LDS(PREP_SUMS, 0);
    SEG_GROUP_LIGHT(sg);
    const KConst kc = cd.kc;
    const sph_params& pr = cd.pr;
    const PView S = cd.S;
    const QView Q = cd.Q;
    if (S.i_type[i] > 2) return;
    if (S.p_type[i] >= 1000) return;
    if (S.p_type[i] <= 0) return;
    const double ki = fmax(S.k_turb[i], 0.0), nui = S.vis_t[i];
    const double gc11 = Q.inv_xx[i], gc12 = Q.inv_xy[i], gc22 = Q.inv_yy[i];
    const double gc23 = Q.inv_yz[i], gc31 = Q.inv_zx[i], gc33 = Q.inv_zz[i];
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    const double uxi = S.ux[i], uyi = S.uy[i], uzi = S.uz[i];
    const double hi = S.h[i], tmp_A = calc_tmpA<double>(kc, hi);
    const bool filt = (cd.count % pr.freq_filt) == 0;
    const bool les = (pr.fv_solve != 0) && (pr.turbulence_model != SPH_LAMINAR);
    OrderedSums<PREP_SUMS, GROUP> sums(wlds_);   // st11, 12, 22, 23, 31, 33, filter, sigma
    const NLRow row = nl_row(cd.nl, i);
    for (int k = g_; k - g_ < row.cnt; k += GROUP) {
        const unsigned e = k < row.cnt ? NB_AT(row, k) : 0u;
        const bool pair = (e & F_HP) != 0;
        if (!__any(pair)) continue;
        double v[PREP_SUMS] = {};
        if (pair) {
            const int j = e & NB_IDX;
            const double dx = xi - S.x[j], dy = yi - S.y[j], dz = zi - S.z[j];
            const double mj = S.m[j], rhoj = S.rho[j];
            const double tdist = sqrt(dx * dx + dy * dy + dz * dz) + 1e-20;
            const double tmp_wij = kernel_w<double>(kc, tmp_A, hi, tdist);
            if (filt) v[6] = mj / rhoj * tmp_wij;
            if (les) {
                v[7] = tdist * tdist * tmp_wij * mj / rhoj;
                if (S.p_type[j] == 1) {
                    const double tmp_dwij = kernel_dw<double>(kc, tmp_A, hi, tdist);
                    const double tdwx = tmp_dwij * dx / tdist;
                    const double tdwy = tmp_dwij * dy / tdist;
                    const double tdwz = tmp_dwij * dz / tdist;
                    const double tdwxc = gc11 * tdwx + gc12 * tdwy + gc31 * tdwz;
                    const double tdwyc = gc12 * tdwx + gc22 * tdwy + gc23 * tdwz;
                    const double tdwzc = gc31 * tdwx + gc23 * tdwy + gc33 * tdwz;
                    const double dux = S.ux[j] - uxi, duy = S.uy[j] - uyi, duz = S.uz[j] - uzi;
                    v[0] = mj / rhoj * dux * tdwxc;
                    v[1] = 0.5 * mj / rhoj * (dux * tdwyc + duy * tdwxc);
                    v[2] = mj / rhoj * duy * tdwyc;
                    v[3] = 0.5 * mj / rhoj * (duy * tdwzc + duz * tdwyc);
                    v[4] = 0.5 * mj / rhoj * (dux * tdwzc + duz * tdwxc);
                    v[5] = mj / rhoj * duz * tdwzc;
                }
            }
        }
        sums.add(v);
    }
    double t[PREP_SUMS];
    for (int a = 0; a < PREP_SUMS; a++) t[a] = sums.sum(a);
    if (g_ == 0) prep_store(cd, i, les, filt, ki, nui, hi, t[6], t[7], t[0], t[1], t[2], t[3], t[4], t[5]);
}

// MIXED passes over the neighbours of particle i: the pair arithmetic in
// float, the sums in double.  REC: the pair's fields come from the compact
// records (float positions, whose float difference is the rounded exact
// difference), else from the field arrays (prep, which runs before the
// double records are packed) or those records.
template <bool REC, class Src, int W>
__device__ __forceinline__ void prep_sums(const CaseDesc& cd, int i, const NLRow row, const Src src, int g, bool filt,
                                          bool les, double& flt, double& sigma, double (&st)[6]) {
    const KConst kc = cd.kc;
    const PView S = cd.S;
    const QView Q = cd.Q;
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    const float xf = (float)xi, yf = (float)yi, zf = (float)zi;
    const double uxi = S.ux[i], uyi = S.uy[i], uzi = S.uz[i];
    const float gc11 = (float)Q.inv_xx[i], gc12 = (float)Q.inv_xy[i], gc22 = (float)Q.inv_yy[i];
    const float gc23 = (float)Q.inv_yz[i], gc31 = (float)Q.inv_zx[i], gc33 = (float)Q.inv_zz[i];
    const float hi = (float)S.h[i], tmp_A = calc_tmpA<float>(kc, hi), f = dw_factor<float>(kc, hi);
    const HScale hs(kc, hi);
    // consecutive neighbours mostly share rho: its reciprocal is kept
    float rho_c = NO_VALUE, yrho = 0.0f;
    walk_row<REC, 2, 2, W>(row, src, g, [&](unsigned e, const Pieces<2, 2>& rec_) {
        if (!(e & F_HP)) return;
        const int j = e & NB_IDX;
        float dx, dy, dz, mj, rhoj, dux, duy, duz;
        int ptj;
        if constexpr (REC) {
            // (every piece is read here: see walk_row)
            const rec_f4 a = rec_.f[0], b = rec_.f[1];
            const rec_d2 p = rec_.d[0], q = rec_.d[1];
            dux = (float)(p.x - uxi); duy = (float)(p.y - uyi); duz = (float)(q.x - uzi);
            dx = xf - a.x; dy = yf - a.y; dz = zf - a.z; mj = a.w; rhoj = b.x;
            ptj = crec_ptype(b.w);
        } else {
            dx = (float)(xi - S.x[j]); dy = (float)(yi - S.y[j]); dz = (float)(zi - S.z[j]);
            mj = (float)S.m[j]; rhoj = (float)S.rho[j];
            ptj = S.p_type[j];
        }
        if (rhoj != rho_c) { rho_c = rhoj; yrho = recip(rhoj); }
        const Dist d = dist_of(dx * dx + dy * dy + dz * dz);
        const float tR = hs.tR(d.r);
        const float wij = kernel_w_t<float>(kc, tmp_A, tR);
        const float vj = quot_any(mj, rhoj, yrho);
        if (filt) flt += (double)(vj * wij);
        if (les) {
            sigma += (double)quot_any(d.r * d.r * wij * mj, rhoj, yrho);
            if (ptj == 1) {
                if constexpr (!REC) {
                    dux = (float)(S.ux[j] - uxi); duy = (float)(S.uy[j] - uyi); duz = (float)(S.uz[j] - uzi);
                }
                const float dw = kernel_dw_t<float>(kc, tmp_A, f, tR);
                const float tx = quot(dw * dx, d.r, d.y), ty = quot(dw * dy, d.r, d.y), tz = quot(dw * dz, d.r, d.y);
                const float cx = gc11 * tx + gc12 * ty + gc31 * tz, cy = gc12 * tx + gc22 * ty + gc23 * tz,
                            cz = gc31 * tx + gc23 * ty + gc33 * tz;
                st[0] += (double)(vj * dux * cx);
                st[1] += (double)(0.5f * vj * (dux * cy + duy * cx));
                st[2] += (double)(vj * duy * cy);
                st[3] += (double)(0.5f * vj * (duy * cz + duz * cy));
                st[4] += (double)(0.5f * vj * (dux * cz + duz * cx));
                st[5] += (double)(vj * duz * cz);
            }
        }
    });
}
template <class Src, int W = 1>
__device__ __forceinline__ void prep_mixed(const CaseDesc& cd, int i, const NList& nl, int li, const Src src,
                                           int g = 0) {
    const sph_params& pr = cd.pr;
    const PView S = cd.S;
    if (S.i_type[i] > 2) return;
    if (S.p_type[i] >= 1000) return;
    if (S.p_type[i] <= 0) return;
    const bool filt = (cd.count % pr.freq_filt) == 0;
    const bool les = (pr.fv_solve != 0) && (pr.turbulence_model != SPH_LAMINAR);
    double flt = 0.0, sigma = 0.0, st[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const NLRow row = nl_row(nl, li);
    if constexpr (Src::lds) {
        prep_sums<true, Src, W>(cd, i, row, src, g, filt, les, flt, sigma, st);
    } else {
        if (src.ok()) prep_sums<true, Src, W>(cd, i, row, src, g, filt, les, flt, sigma, st);
        else prep_sums<false, Src, W>(cd, i, row, src, g, filt, les, flt, sigma, st);
    }
    if constexpr (W > 1) {
        group_fold<W>(flt); group_fold<W>(sigma);
        for (double& v : st) group_fold<W>(v);
        if (g != 0) return;
    }
    prep_store(cd, i, les, filt, fmax(S.k_turb[i], 0.0), S.vis_t[i], S.h[i], flt, sigma, st[0], st[1], st[2], st[3],
               st[4], st[5]);
}
__global__ void __launch_bounds__(MAX_BLOCK) k_prep_mixed(Seg sg) {
    SEG_GROUP_LIGHT(sg);
    prep_mixed<GSrc, GROUP>(cd, i, cd.nl, i, GSrc{&cd.crec_adv, (size_t)cd.n}, g_);
}
__global__ void __launch_bounds__(WAVE_BLOCK) k_prep_heavy(Seg sg) {
    SEG_HEAVY(sg);
    prep_mixed<GSrc, 64>(cd, i, cd.nl, i, GSrc{&cd.crec_adv, (size_t)cd.n}, lane_);
}
__global__ void __launch_bounds__(TILE_THREADS) k_prep_tile(Seg sg, int width) {
    TILE_CHUNK(sg, width, cd.crec_adv, CREC_ADV_FLOATS);
    TILE_LANES(width) {
        if (chunk_.y >= 0) prep_mixed<LSrc<CREC_ADV_FLOATS>, GROUP>(cd, i, cd.tile.nl, lane_, TILE_SRC(CREC_ADV_FLOATS), g_);
        else prep_mixed<GSrc, GROUP>(cd, i, cd.tile.nl, lane_, GSrc{&cd.crec_adv, (size_t)cd.n}, g_);
    }
}

// ------------------------------------------------------------------------
// KERNEL_boundary3D, functions_BC.cuh:100-190 (wall velocity)
constexpr int BD_SUMS = 4;
__global__ void __launch_bounds__(WAVE_BLOCK) k_boundary3d(Seg sg) {
    __shared__ double lds[WAVE_BLOCK / 64][ord_doubles(BD_SUMS)];
    SEG_BOUNDARY(sg);
    const sph_params& pr = cd.pr;
    if (pr.noslip_bc != 1) return;   // ISPH_Calc.cuh:83
    const PView S = cd.S;
    if (S.i_type[i] > 2) return;
    if (S.p_type[i] != 0) return;
    const KConst kc = cd.kc;
    const double hi = S.h[i], tmp_A = calc_tmpA<double>(kc, hi);
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    OrderedSums<BD_SUMS, BLANES> sums(lds[threadIdx.x >> 6]);
    if (lane == 3) sums.acc = 1.0e-10;   // the weights' sum
    const NLRow row = nl_row(cd.nl, i);
    for (int k = lane; k - lane < row.cnt; k += BLANES) {
        const unsigned e = k < row.cnt ? NB_AT(row, k) : 0u;
        const int j = e & NB_IDX;
        double v[BD_SUMS] = {};
        if (e & F_HM) {
            const int p_type_j = S.p_type[j];
            if ((p_type_j > 0) && (p_type_j != 9)) {
                const double dx = xi - S.x[j], dy = yi - S.y[j], dz = zi - S.z[j];
                const double tdist = sqrt(dx * dx + dy * dy + dz * dz) - 1e-20;
                const double twij = kernel_w<double>(kc, tmp_A, hi, tdist);
                v[0] = S.ux[j] * twij;
                v[1] = S.uy[j] * twij;
                v[2] = S.uz[j] * twij;
                v[3] = twij;
            }
        }
        sums.add(v);
    }
    double t[BD_SUMS];
    for (int a = 0; a < BD_SUMS; a++) t[a] = sums.sum(a);
    if (lane != 0) return;
    const double uxi = S.ux[i], uyi = S.uy[i], uzi = S.uz[i];
    S.ux[i] = 2 * uxi * 0 - t[0] / t[3];
    S.uy[i] = 2 * uyi * 0 - t[1] / t[3];
    S.uz[i] = 2 * uzi * 0 - t[2] / t[3];
}

// The same in MIXED: lane sums over entries lane, lane + BLANES, ..., then a
// fixed butterfly, so a case gives the same bits alone and in a batch; only
// the particles the reference's kernel writes (p_type 0 and 9) are visited.
__global__ void __launch_bounds__(WAVE_BLOCK) k_boundary3d_mixed(Seg sg) {
    SEG_BOUNDARY(sg);
    const sph_params pr = cd.pr;
    if (pr.noslip_bc != 1) return;   // ISPH_Calc.cuh:83
    const PView S = cd.S;
    if (S.i_type[i] > 2) return;
    const int p_type_i = S.p_type[i];
    if (p_type_i != 0 && p_type_i != 9) return;
    const KConst kc = cd.kc;
    const NList nl = cd.nl;
    const float hi = (float)S.h[i], tmp_A = calc_tmpA<float>(kc, hi);
    const HScale hs(kc, hi);
    double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    const NLRow row = nl_row(nl, i);
    for (int k = lane; k < row.cnt; k += BLANES) {
        unsigned e = NB_AT(row, k);
        if (!(e & F_HM)) continue;
        int j = e & NB_IDX;
        const int p_type_j = S.p_type[j];
        if (!((p_type_j > 0) && (p_type_j != 9))) continue;
        float dx = (float)(xi - S.x[j]), dy = (float)(yi - S.y[j]), dz = (float)(zi - S.z[j]);
        const float twij = kernel_w_t<float>(kc, tmp_A, hs.tR(dist_of(dx * dx + dy * dy + dz * dz).r));
        t[0] += (double)((float)S.ux[j] * twij);
        t[1] += (double)((float)S.uy[j] * twij);
        t[2] += (double)((float)S.uz[j] * twij);
        t[3] += (double)twij;
    }
    for (double& v : t) group_fold<BLANES>(v);
    if (lane != 0) return;
    const double flt = 1.0e-10 + t[3];
    const double uxi = S.ux[i], uyi = S.uy[i], uzi = S.uz[i];
    S.ux[i] = 2 * uxi * (p_type_i == 9) - t[0] / flt;
    S.uy[i] = 2 * uyi * (p_type_i == 9) - t[1] / flt;
    S.uz[i] = 2 * uzi * (p_type_i == 9) - t[2] / flt;
}

// ------------------------------------------------------------------------
// KERNEL_MOST_boundary3D, functions_MOST.cuh:175-322.  Part 1: the
// surface-layer fluxes of each MOST particle; the neighbour heat deposit is
// stored per particle for the gather in part 2.
__global__ void __launch_bounds__(MAX_BLOCK) k_most_self(Seg sg) {
    SEG_PARTICLE(sg);
    const sph_params pr = cd.pr;
    const PView S = cd.S;
    double* dep = cd.snap[4];   // the snapshots are not live between the copy passes
    const int count = cd.count;
    const double dt = cd.dt;
    if (S.MOST_buffer[i] != 1) { dep[i] = 0.0; return; }
    const double KVK = 0.4;
    double zi = S.z[i];
    double uxi = S.ux[i], uyi = S.uy[i];
    double tempi = S.temp[i], rhoi = S.rho[i], mi = S.m[i];
    double space = S.h[i] / 1.5;
    double z0 = pr.most_z0, z0h = pr.most_z0h;
    double u_star = 0.0, theta_star = 0.0, OB_length;
    double theta_surface = wall_temperature(pr, dt, count);
    double wind_speed = sqrt(uxi * uxi + uyi * uyi);
    wind_speed = fmax(0.001, fmin(wind_speed, 100.0));
    if (pr.most_mode == SPH_MOST_PRESCRIBED_L) {
        OB_length = pr.most_L;
        u_star = KVK * wind_speed / Phi_m(OB_length, zi, z0);
        theta_star = KVK * (tempi - theta_surface) / Phi_h(OB_length, zi, z0h);
    } else {
        double Ri_b = (pr.gravity / tempi) * (tempi - theta_surface) * zi / (wind_speed * wind_speed + 1e-10);
        if (fabs(Ri_b) > 1e-3) {
            OB_length = zi / Ri_b;
            OB_length = fmax(-500.0, fmin(OB_length, 500.0));
            for (int iter = 0; iter < 200; iter++) {
                double ol_m = OB_length, ol_l = 0.999 * ol_m, ol_u = 1.001 * ol_m;
                double pm = Phi_m(ol_m, zi, z0);
                double fL = Ri_b - (zi / ol_m) * Phi_h(ol_m, zi, z0h) / (pm * pm);
                double dfL = ((-(zi / ol_u) * Phi_h(ol_u, zi, z0h) / (Phi_m(ol_u, zi, z0) * Phi_m(ol_u, zi, z0))) -
                              (-(zi / ol_l) * Phi_h(ol_l, zi, z0h) / (Phi_m(ol_l, zi, z0) * Phi_m(ol_l, zi, z0)))) /
                             (ol_u - ol_l);
                OB_length -= 1.0 * fL / dfL;
                if (fabs(OB_length) > 1e-6) {
                    if (fabs((OB_length - ol_m) / OB_length) < 1e-5) break;
                    else if (fabs(OB_length - ol_m) < 1e-5) break;
                }
            }
            u_star = KVK * wind_speed / Phi_m(OB_length, zi, z0);
            theta_star = KVK * (tempi - theta_surface) / Phi_h(OB_length, zi, z0h);
        } else {
            OB_length = 1e6;
            u_star = KVK * wind_speed / log(zi / z0);
            theta_star = KVK * (tempi - theta_surface) / log(zi / z0h);
        }
    }
    double momentum_x = -rhoi * u_star * (uxi * u_star / wind_speed);
    double momentum_y = -rhoi * u_star * (uyi * u_star / wind_speed);
    double shf = -rhoi * pr.air_cp * u_star * theta_star * 100.0;
    dep[i] = 0.5 * shf / (space * rhoi * pr.air_cp);
    S.fmx[i] = 1.0 * momentum_x * space * space / mi;
    S.fmy[i] = 1.0 * momentum_y * space * space / mi;
    S.float1[i] = u_star; S.float2[i] = theta_star; S.float3[i] = OB_length;
}

// Part 2: every particle j gathers the deposits of the MOST particles i whose
// ghost node (x_i, y_i, z_i + dz) lies within ghost_r of j and whose 3x3x3
// ghost window holds j's cell, in ascending i, with i's own deposit applied
// after its neighbour deposits (functions_MOST.cuh:286-316 serialised).
__global__ void __launch_bounds__(MAX_BLOCK) k_most_deposit(Seg sg) {
    SEG_PARTICLE(sg);
    const int j = i;
    const sph_params pr = cd.pr;
    const PView S = cd.S;
    const QView Q = cd.Q;
    const Grid g = cd.g;
    const double* dep = cd.snap[4];
    const int* keys = cd.keys;
    const sph_domain& d = g.d;
    const bool self_most = S.MOST_buffer[j] == 1;
    double xj = S.x[j], yj = S.y[j], zj = S.z[j];
    double acc = 0.0, last = 0.0;
    bool any = false, self_done = !self_most;
    int key_j = keys[j];
    int cj_i = key_j % d.NI, cj_j = (key_j / d.NI) % d.NJ, cj_k = key_j / (d.NI * d.NJ);
    double r = pr.most_ghost_r;
    double px = xj, py = yj, pz = zj - pr.most_ghost_dz;
    double mg = 1e-6 + 1e-6 * r;
    bool box_ok = !(pz + r + mg < (double)d.z_min || pz - r - mg > (double)d.z_max ||
                    px + r + mg < (double)d.x_min || px - r - mg > (double)d.x_max ||
                    py + r + mg < (double)d.y_min || py - r - mg > (double)d.y_max);
    if (box_ok && key_j < d.num_cells - 1) {
        int i0 = bin_axis((float)(px - r - mg), d.x_min, d.x_max, d.NI), i1 = bin_axis((float)(px + r + mg), d.x_min, d.x_max, d.NI);
        int j0 = bin_axis((float)(py - r - mg), d.y_min, d.y_max, d.NJ), j1 = bin_axis((float)(py + r + mg), d.y_min, d.y_max, d.NJ);
        int k0 = bin_axis((float)(pz - r - mg), d.z_min, d.z_max, d.NK), k1 = bin_axis((float)(pz + r + mg), d.z_min, d.z_max, d.NK);
        for (int ck = k0; ck <= k1; ck++)
            for (int cj = j0; cj <= j1; cj++)
                for (int ci = i0; ci <= i1; ci++) {
                    int cell = ci + d.NI * cj + d.NI * d.NJ * ck;
                    int s = g.gstr[cell];
                    if (s == -1) continue;
                    int e = g.gend[cell];
                    for (int i = s; i < e; i++) {
                        if (!self_done && i > j) { acc += dep[j]; last = dep[j]; any = true; self_done = true; }
                        if (S.MOST_buffer[i] != 1) continue;
                        double xg = S.x[i], yg = S.y[i], zg = S.z[i] + pr.most_ghost_dz;
                        Cell c = query_cell(d, xg, yg, zg);
                        bool inwin = abs(cj_i - c.i) <= 1 && abs(cj_j - c.j) <= 1 && abs(cj_k - c.k) <= 1;
                        double tdist = dist3<double>(xg, yg, zg, xj, yj, zj) - 1e-20;
                        if (inwin && tdist < pr.most_ghost_r) { acc += dep[i]; last = dep[i]; any = true; }
                        if (i == j) { acc += dep[j]; last = dep[j]; any = true; self_done = true; }
                    }
                }
    }
    if (!self_done) { acc += dep[j]; last = dep[j]; any = true; }
    if (any) { Q.dtemp[j] += acc; S.hmz[j] = last; }
}

// ------------------------------------------------------------------------
// KERNEL_Neumann_boundary3D, functions_BC.cuh:290-446.  Pressures are read
// from a snapshot (pold) taken before the launch.
// The window of the Neumann scan around cell c (ncell nc), in scan order
// (z-major rows of x-cells, the particles of a row in sorted order), as
// chunks of 64 candidates: f(j, count) with lane l holding candidate l of
// the chunk (j < 0: none) and count the chunk's candidates.  Every lane
// makes the same calls.
template <class F>
__device__ __forceinline__ void neumann_window(const Grid& g, const Cell& c, int nc, int lane, F&& f) {
    const int side = 2 * nc + 1, nrows = side * side;
    if (nrows <= 64) {
        // Lane k holds x-row k of the window (z-major, then y): its particle
        // range and the exclusive prefix of the lengths, so the window's
        // candidates are numbered v = 0 .. total-1 in scan order.
        int rs = 0, rl = 0;
        if (lane < nrows) {
            int2 rg;
            if (row_range(g, c.i - nc, c.i + nc, c.j + lane % side - nc, c.k + lane / side - nc, rg)) {
                rs = rg.x;
                rl = rg.y - rg.x;
            }
        }
        int incl = rl;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(incl, off, 64);
            if (lane >= off) incl += o;
        }
        const int excl = incl - rl, total = __shfl(incl, 63, 64);
        for (int v0 = 0; v0 < total; v0 += 64) {
            const int v = v0 + lane, vv = min(v, total - 1);
            // the row holding vv: the last row whose prefix is <= vv (never
            // an empty row); every lane takes part in every shuffle
            int lo = 0;
#pragma unroll
            for (int step = 32; step > 0; step >>= 1) {
                const int cand = lo + step;
                const int pe = __shfl(excl, min(cand, 63), 64);
                if (cand < nrows && pe <= vv) lo = cand;
            }
            const int start = __shfl(rs, lo, 64), pre = __shfl(excl, lo, 64);
            f(v < total ? start + (vv - pre) : -1, min(64, total - v0));
        }
    } else {
        for (int z = -nc; z <= nc; z++)
            for (int y = -nc; y <= nc; y++) {
                int2 rg;
                if (!row_range(g, c.i - nc, c.i + nc, c.j + y, c.k + z, rg)) continue;
                for (int b = rg.x; b < rg.y; b += 64) f(b + lane < rg.y ? b + lane : -1, min(64, rg.y - b));
            }
    }
}

// Neumann pairs of one boundary particle per 64-thread block: the
// candidates of its window that carry weight in the Neumann sums (fluid,
// non-buffer, inside the 2h search range, with the pass's own precision R
// for the distance), in scan order.  COUNT: their number; FILL: the list.
template <class R, bool FILL>
__global__ void __launch_bounds__(64) k_nmp_build(PView A, Grid g, KConst kc, double L2, const int* nm_list,
                                                  int nm_count, int* cnt, const long long* off, int* ent) {
    const int u = blockIdx.x, lane = threadIdx.x;
    if (u >= nm_count) return;
    const int i = nm_list[u];
    const R hi = (R)(2.0 * A.h[i]);
    const R search_range = (R)kc.kappa * hi;
    const double xi = A.x[i], yi = A.y[i], zi = A.z[i];
    const int bt = A.buffer_type[i];
    const double xg = (bt == 1 || bt == -1) ? 2.0 * L2 - xi : xi;
    const Cell c = query_cell(g.d, xg, yi, zi);
    const long long at = FILL ? off[u] : 0;
    int n = 0;
    neumann_window(g, c, A.ncell[i], lane, [&](int j, int count) {
        (void)count;
        bool hit = false;
        if (j >= 0 && A.p_type[j] == 1 && A.buffer_type[j] == 0) {
            R dx = (R)(xg - A.x[j]), dy = (R)(yi - A.y[j]), dz = (R)(zi - A.z[j]);
            R tdist = sqrt(dx * dx + dy * dy + dz * dz) - (R)1e-20;
            hit = tdist < search_range;
        }
        const unsigned long long m = __ballot(hit);
        if (FILL && hit) ent[at + n + __popcll(m & ((1ULL << lane) - 1ULL))] = j;
        n += __popcll(m);
    });
    if (!FILL && lane == 0) cnt[u] = n;
}
__global__ void __launch_bounds__(BLOCK) k_nmp_widen(int n, const int* a, long long* b) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r < n) b[r] = a[r];
}

// FP64: a 64-lane wave per boundary particle of the case's compact list, over
// its listed pairs.  Each lane forms the terms of one pair exactly as a serial
// scan does, and the sums are added in list order (OrderedSums).  (Each lane
// adding the terms that a flag marked, one LDS read after another, took half of
// the pass: 268 us on a 150 k canyon.)
constexpr int NM_BLOCK = 64;
__global__ void __launch_bounds__(NM_BLOCK) k_neumann(Seg sg, int which, int only_count0) {
    int first_;
    const int cid_ = seg_case(sg, first_);
    const CaseDesc& cd = sg.cd[cid_];
    const int u = first_ >> 6, lane = threadIdx.x;
    if (u >= cd.nm_count) return;
    if (only_count0 && cd.count != 0) return;   // the extra pre-advection call, ISPH_Calc.cuh:88-90
    const KConst kc = cd.kc;
    const sph_params pr = cd.pr;
    const PView A = which ? cd.P : cd.S;
    const Grid g = cd.g;
    const double* pold = cd.snap[3];
    const int i = cd.nm_list[u];
    const double hi = 2.0 * A.h[i], tmp_A = calc_tmpA<double>(kc, hi), search_range = kc.kappa * hi;
    const double xi = A.x[i], yi = A.y[i], zi = A.z[i];
    double pres_g = 0;
    const int bt = A.buffer_type[i];
    // the ghost pressure and the gradient only enter the inlet formula
    const bool inlet = (bt == 1 || bt == -1);
    const double xg = inlet ? 2.0 * pr.L2 - xi : xi, yg = yi, zg = zi;
    const Cell c = query_cell(g.d, xg, yg, zg);
    // The window's cells of one x-row are consecutive in cell order, so
    // their particles form one range of the sorted order, visited in the
    // same order as cell by cell.  Lanes test consecutive candidates; the
    // last match in that order wins, as in the serial scan.
    for (int z = -1; z <= 1 && inlet; z++)
        for (int y = -1; y <= 1; y++) {
            int2 rg;
            if (!row_range(g, c.i - 1, c.i + 1, c.j + y, c.k + z, rg)) continue;
            for (int b = rg.x; b < rg.y; b += 64) {
                const int j = b + lane;
                bool hit = false;
                double pj = 0.0;
                if (j < rg.y) {
                    const double dx = xg - A.x[j], dy = yg - A.y[j], dz = zg - A.z[j];
                    const double dist = sqrt(dx * dx + dy * dy + dz * dz) - 1e-20;
                    hit = dist < pr.neumann_ghost_r;
                    pj = pold[j];
                }
                const unsigned long long m = __ballot(hit);
                if (m) pres_g = __shfl(pj, 63 - __clzll(m), 64);
            }
        }
    __shared__ double terms[ord_doubles(8)];
    OrderedSums<8, 64> sums(terms);
    // (only fluid, non-buffer neighbours carry weight: the reference
    // multiplies the others by 0, and leaving those exact zeros out of the
    // list leaves every sum bit for bit the same)
    const long long e0 = cd.nmp_off[u], e1 = cd.nmp_off[u + 1];
    for (long long b = e0; b < e1; b += 64) {
        double v[8] = {};
        if (b + lane < e1) {
            const int j = cd.nmp_ent[b + lane];
            const double dx = xg - A.x[j], dy = yg - A.y[j], dz = zg - A.z[j];
            const double tdist = sqrt(dx * dx + dy * dy + dz * dz) - 1e-20;
            if (tdist < search_range) {
                const double mj = A.m[j], rhoj = A.rho[j];
                const double presj = pold[j];
                const double twij = kernel_w<double>(kc, tmp_A, hi, tdist);
                v[0] = mj / rhoj * presj * twij;
                v[1] = mj / rhoj * A.ux[j] * twij;
                v[2] = mj / rhoj * A.uy[j] * twij;
                v[3] = mj / rhoj * A.uz[j] * twij;
                v[4] = mj / rhoj * twij;
                if (inlet) {
                    const double tdwij = kernel_dw<double>(kc, tmp_A, hi, tdist);
                    const double tdwx = dx / tdist * tdwij, tdwy = dy / tdist * tdwij, tdwz = dz / tdist * tdwij;
                    const double dp = presj - pres_g;
                    v[5] = mj / rhoj * dp * tdwx;
                    v[6] = mj / rhoj * dp * tdwy;
                    v[7] = mj / rhoj * dp * tdwz;
                }
            }
        }
        sums.add(v);
    }
    const double tpres = sums.sum(0), tux = sums.sum(1), tuy = sums.sum(2), tuz = sums.sum(3), tflt_s = sums.sum(4);
    const double grad_px = sums.sum(5), grad_py = sums.sum(6), grad_pz = sums.sum(7);
    if (lane != 0) return;
    if (tflt_s < 1e-6) {
        A.pres[i] = 0.0;
    } else {
        A.pres[i] = tpres / tflt_s;
        if (A.p_type[i] == -1) { A.ux[i] = tux / tflt_s; A.uy[i] = tuy / tflt_s; A.uz[i] = tuz / tflt_s; }
        if (inlet) A.pres[i] = pres_g + (xi - xg) * grad_px + (yi - yg) * grad_py + (zi - zg) * grad_pz;
    }
}

// The listed pairs of one boundary particle (nm_cent or particle numbers) as
// a row of entries for walk_row; every entry counts.
struct NMRow {
    const int* p;
    int cnt;
    __device__ unsigned at(int k) const {
        return (unsigned)((const __attribute__((address_space(1))) int*)p)[k] | F_DP;
    }
};
// MIXED: NM_LANES lanes a boundary particle, each adding the
// terms of pairs lane, lane + NM_LANES, ... in list order, then a fixed butterfly
// (so the sums are the same on every call, alone or in a batch).  A wave a
// particle spent most of its time on the loads before its few rounds.  By lanes
// (64 without the pipelined walk, 32, 16): 374, 273, 238 us on the 2.13 M canyon,
// 91, 67, 63 on 200 k, 20.6, 19.3, 24.3 on 20 k, 171, 198, 355 on a refined canyon,
// whose 329 markers have thousands of pairs.
constexpr int NM_LANES = 32;
__global__ void __launch_bounds__(WAVE_BLOCK) k_neumann_mixed(Seg sg, int which, int only_count0) {
    SEG_BOUNDARY_LANES(sg, NM_LANES);
    if (only_count0 && cd.count != 0) return;   // the extra pre-advection call, ISPH_Calc.cuh:88-90
    const KConst kc = cd.kc;
    const sph_params& pr = cd.pr;
    const PView A = which ? cd.P : cd.S;
    const Grid g = cd.g;
    const double* const pold = cd.snap[3];
    const float hi = (float)(2.0 * A.h[i]), tmp_A = calc_tmpA<float>(kc, hi);
    const double xi = A.x[i], yi = A.y[i], zi = A.z[i];
    const int bt = A.buffer_type[i];
    const bool inlet = (bt == 1 || bt == -1);
    const double xg = inlet ? 2.0 * pr.L2 - xi : xi;
    double pres_g = 0;
    if (inlet) {   // the ghost pressure: see k_neumann
        const Cell c = query_cell(g.d, xg, yi, zi);
        const int first = (int)(threadIdx.x & 63) & ~(NM_LANES - 1);
        for (int z = -1; z <= 1; z++)
            for (int y = -1; y <= 1; y++) {
                int2 rg;
                if (!row_range(g, c.i - 1, c.i + 1, c.j + y, c.k + z, rg)) continue;
                for (int b = rg.x; b < rg.y; b += NM_LANES) {
                    const int j = b + lane;
                    bool hit = false;
                    double pj = 0.0;
                    if (j < rg.y) {
                        const float dx = (float)(xg - A.x[j]), dy = (float)(yi - A.y[j]), dz = (float)(zi - A.z[j]);
                        const float dist = sqrt(dx * dx + dy * dy + dz * dz) - 1e-20f;
                        hit = dist < (float)pr.neumann_ghost_r;
                        pj = pold[j];
                    }
                    const unsigned m = (unsigned)(__ballot(hit) >> first) & ((unsigned)(~0ULL >> (64 - NM_LANES)));
                    if (m) pres_g = __shfl(pj, first + 31 - __clz((int)m), 64);
                }
            }
    }
    const HScale hs(kc, hi);
    const float dwf = dw_factor<float>(kc, hi);
    float rho_c = NO_VALUE, yrho = 0.0f;
    double s[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    auto add = [&](float dx, float dy, float dz, float mj, float rhoj, float uxj, float uyj, float uzj, double presj) {
        if (rhoj != rho_c) { rho_c = rhoj; yrho = recip(rhoj); }
        // (the list holds exactly the pairs inside the search range)
        const Dist d = dist_of(dx * dx + dy * dy + dz * dz);
        const float tR = hs.tR(d.r), w = kernel_w_t<float>(kc, tmp_A, tR), vj = quot_any(mj, rhoj, yrho);
        s[0] += (double)(vj * (float)presj * w);
        s[1] += (double)(vj * uxj * w);
        s[2] += (double)(vj * uyj * w);
        s[3] += (double)(vj * uzj * w);
        s[4] += (double)(vj * w);
        if (inlet) {
            const float dw = kernel_dw_t<float>(kc, tmp_A, dwf, tR), dp = vj * (float)(presj - pres_g);
            s[5] += (double)(dp * (quot(dx, d.r, d.y) * dw));
            s[6] += (double)(dp * (quot(dy, d.r, d.y) * dw));
            s[7] += (double)(dp * (quot(dz, d.r, d.y) * dw));
        }
    };
    const long long e0 = cd.nmp_off[u_];
    const int cnt = (int)(cd.nmp_off[u_ + 1] - e0);
    if (cd.nm_rec) {   // packed, with float-exact positions (see walk_row)
        const GSrc src{&cd.nm_rec, (size_t)cd.nm_nset};
        walk_row<true, 2, 1, NM_LANES>(NMRow{cd.nmp_cent + e0, cnt}, src, lane, [&](unsigned e, const Pieces<2, 1>& r) {
            const rec_f4 a = r.f[0], b = r.f[1];
            const float dx = (float)(xg - (double)a.x), dy = (float)(yi - (double)a.y), dz = (float)(zi - (double)a.z);
            const double presj = r.d[0].x;
            if (e) add(dx, dy, dz, a.w, b.x, b.y, b.z, b.w, presj);
        });
    } else {
        walk_row<false, 1, 0, NM_LANES>(NMRow{cd.nmp_ent + e0, cnt}, 0, lane, [&](unsigned e, const Pieces<1, 0>&) {
            if (!e) return;
            const int j = (int)(e & NB_IDX);
            add((float)(xg - A.x[j]), (float)(yi - A.y[j]), (float)(zi - A.z[j]), (float)A.m[j], (float)A.rho[j],
                (float)A.ux[j], (float)A.uy[j], (float)A.uz[j], pold[j]);
        });
    }
    for (double& v : s) group_fold<NM_LANES>(v);
    if (lane != 0) return;
    const double tflt = s[4];
    if (tflt < 1e-6) {
        A.pres[i] = 0.0;
    } else {
        A.pres[i] = s[0] / tflt;
        if (A.p_type[i] == -1) { A.ux[i] = s[1] / tflt; A.uy[i] = s[2] / tflt; A.uz[i] = s[3] / tflt; }
        if (inlet) A.pres[i] = pres_g + (xi - xg) * s[5] + 0.0 * s[6] + 0.0 * s[7];
    }
}

// ------------------------------------------------------------------------
// KERNEL_advection_force3D, functions_PPE.cuh:191-480
// SCAL: some case of the launch transports temperature or concentration or
// uses the Boussinesq buoyancy; without them (the canyon) those terms and
// their registers are compiled out (130 -> fewer VGPRs, more waves per SIMD)
struct AdvSums {   // viscous and artificial (t), convective (c) terms; scalars
    double tx = 0, ty = 0, tz = 0, cx = 0, cy = 0, cz = 0, rc = 0, rd = 0, ct = 0, temp = 0, flt = 0;
};
__device__ __forceinline__ void advection_store(const CaseDesc& cd, int i, const AdvSums& a, bool con_solve,
                                                bool concn_solve, bool boussinesq_solve, double cpi) {
    const sph_params& pr = cd.pr;
    const QView Q = cd.Q;
    const int ptypei = cd.S.p_type[i];
    double tz = a.tz;
    if (pr.fg_solve) tz += -pr.gravity;
    if ((boussinesq_solve) && (ptypei > 0) && (ptypei < 1000))
        tz = 1.0 / pr.T_ini * pr.gravity * (a.temp / a.flt - pr.tempb);
    Q.ftotalx[i] = a.tx - a.cx;
    Q.ftotaly[i] = a.ty - a.cy;
    Q.ftotalz[i] = tz - a.cz;
    if (con_solve) Q.dtemp[i] += a.rc / cpi - a.ct;
    Q.ftotal[i] = sqrt(a.tx * a.tx + a.ty * a.ty + tz * tz);
    if (concn_solve) Q.dconcn[i] = a.rd;
}
// sums tx, ty, tz (a second term each with the artificial viscosity), cx, cy,
// cz and, with SCAL, rc, ct; then rd (two terms), temp, flt
template <bool SCAL> constexpr int adv_sums() { return SCAL ? 8 : 6; }
constexpr int ADV_SECOND = 3, ADV_SUMS2 = 3;
template <bool SCAL>
__global__ void __launch_bounds__(MAX_BLOCK) k_advection(Seg sg) {
    ORDERED_LDS(adv_sums<SCAL>(), ADV_SECOND);
    SEG_GROUP_LIGHT(sg);
    constexpr int NT = adv_sums<SCAL>();
    const KConst kc = cd.kc;
    const sph_params& pr = cd.pr;
    const bool con_solve = SCAL && pr.con_solve, concn_solve = SCAL && pr.concn_solve;
    const bool boussinesq_solve = SCAL && pr.boussinesq_solve;
    const PView S = cd.S;
    if (S.i_type[i] > 2) return;
    const int ptypei = S.p_type[i];
    if (ptypei == 1000) return;
    if (ptypei <= 0) return;
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    const double uxi = S.ux[i], uyi = S.uy[i], uzi = S.uz[i];
    const double tempi = SCAL ? S.temp[i] : 0.0;
    const double hi = S.h[i], mi = S.m[i], rhoi = S.rho[i];
    const double eli = S.eli[i];
    const double tmp_A = calc_tmpA<double>(kc, hi);
    double kci = 0, cpi = 1, concni = 0, diffi = 0;
    if (con_solve) {
        kci = pr.solid_k * (ptypei == 0 || ptypei == 1000) + pr.air_k * (ptypei == 1 || ptypei == -1);
        cpi = pr.solid_cp * (ptypei == 0 || ptypei == 1000) + pr.air_cp * (ptypei == 1 || ptypei == -1);
    }
    if (concn_solve) { concni = S.concn[i]; diffi = pr.diff_coef; }
    const double visi = viscosity2(pr, ptypei) + S.vis_t[i] * S.rho[i];
    const double Alpha = pr.av_alpha, Beta = pr.av_beta, soundspeed = pr.av_c;
    const double ome = 1 - eli;
    const int fv = pr.fv_solve;
    const bool art = pr.artificial_viscosity != 0;
    OrderedSums<NT, GROUP> sums(wlds_);
    OrderedSums<ADV_SUMS2, GROUP> sums2(wlds_);
    const NLRow row = nl_row(cd.nl, i);
    for (int k = g_; k - g_ < row.cnt; k += GROUP) {
        const unsigned e = k < row.cnt ? NB_AT(row, k) : 0u;
        const int j = e & NB_IDX;
        bool pair = (e & F_DP) != 0;
        double hj, vis_tj, xj, yj, zj, mj, uxj, uyj, uzj, rhoj, pqj_;
        int ptypej = 0, itj_;
        if (pair) {
            rec_aux(Rec(cd), j, vis_tj, ptypej, itj_);
            pair = ptypej < 1000;
        }
        if (!__any(pair)) continue;
        double v[NT] = {}, v2[ADV_SECOND] = {}, w[ADV_SUMS2] = {}, w2[1] = {};
        if (pair) {
            rec_pos(Rec(cd), j, xj, yj, zj, mj, rhoj, pqj_);
            rec_vel(Rec(cd), j, uxj, uyj, uzj, hj);
            const double visj = viscosity2(pr, ptypej) + vis_tj * rhoj;
            const double dx = xi - xj, dy = yi - yj, dz = zi - zj;
            const double tdist = sqrt(dx * dx + dy * dy + dz * dz) + 1e-20;
            const double tdwij = kernel_dw<double>(kc, tmp_A, hi, tdist);
            const double tdwx = tdwij * dx / tdist;
            const double tdwy = tdwij * dy / tdist;
            const double tdwz = tdwij * dz / tdist;
            const double dux = uxi - uxj, duy = uyi - uyj, duz = uzi - uzj;   // u_i - u_j
            double tempj = 0.0, concnj = 0.0;
            if (con_solve || concn_solve || boussinesq_solve) rec_scalar(Rec(cd), j, tempj, concnj);
            if (fv == SPH_FV_CLEARY) {
                double C_v = dx * tdwx + dy * tdwy + dz * tdwz;
                C_v *= (visi * visj) / (visi + visj);
                C_v *= 4.0 * (mj / (rhoi * rhoj));
                C_v /= tdist;
                C_v /= tdist;
                v[0] = C_v * dux; v[1] = C_v * duy; v[2] = C_v * duz;
            } else if (fv == SPH_FV_MONAGHAN) {
                double uij_xij = dux * dx + duy * dy + duz * dz;
                double phi_ij = uij_xij;
                phi_ij /= (tdist * tdist + 0.01 * hi * hi);
                double P_ij = -2.0 * (3 + 2.0) * phi_ij * mj / rhoj;
                double C_v = 2.0 * (visi * visj) / (visi + visj - 1e-20);
                double nui = C_v / rhoi;
                P_ij *= nui;
                if (ptypei <= 0 || ptypei >= 1000) P_ij = 0;
                if (ptypej <= 0 || ptypei >= 1000) P_ij = 0;
                v[0] = -(P_ij)*tdwx; v[1] = -(P_ij)*tdwy; v[2] = -(P_ij)*tdwz;
            }
            if (eli < 1.0) {
                const double vx = -dux, vy = -duy, vz = -duz;   // u_j - u_i
                v[3] = (uxi * vx * tdwx + uyi * vx * tdwy + uzi * vx * tdwz) * mj / rhoj * ome;
                v[4] = (uxi * vy * tdwx + uyi * vy * tdwy + uzi * vy * tdwz) * mj / rhoj * ome;
                v[5] = (uxi * vz * tdwx + uyi * vz * tdwy + uzi * vz * tdwz) * mj / rhoj * ome;
                if constexpr (SCAL) {
                    if (con_solve)
                        v[7] = -(2.0 * mj / (rhoi + rhoj) * (tempj - tempi) * (dux * tdwx + duy * tdwy + duz * tdwz) * ome);
                    if (concn_solve) {
                        const double dc = concnj - concni;
                        w[0] = -((uxi * dc * tdwx + uyi * dc * tdwy + uzi * dc * tdwz) * mj / rhoj * ome);
                    }
                }
            }
            if constexpr (SCAL) {
                if (con_solve) {
                    double kcj = pr.solid_k * (ptypej == 0 || ptypej == 1000) + pr.air_k * (ptypej == 1 || ptypej == -1);
                    double rhoj_temp = (ptypej == 1 || ptypej == -1) ? rhoj : pr.solid_rho;
                    double mj_temp = mj * rhoj_temp / rhoj;
                    double sum_con_H = 4.0 * mj_temp * kcj * kci * (tempi - tempj) * tdwij;
                    sum_con_H /= (tdist + 1e-10) * rhoi * rhoj_temp * (kci + kcj);
                    v[6] = sum_con_H;
                }
                if (concn_solve) {
                    double diffj = pr.diff_coef;
                    double tmprd = mi * (diffi * rhoi + diffj * rhoj);
                    tmprd *= (dx * tdwx + dy * tdwy + dz * tdwz);
                    tmprd /= (rhoi * rhoj * (tdist * tdist + 0.01 * hi * hi));
                    w2[0] = tmprd * (concni - concnj) * (double)(ptypei == ptypej);
                }
                if (boussinesq_solve) {
                    const double twij = kernel_w<double>(kc, tmp_A, hi, tdist);
                    w[1] = (mj / rhoj) * tempj * twij;
                    w[2] = (mj / rhoj) * twij;
                }
            }
            if (art) {
                double uij_xij = dux * dx + duy * dy + duz * dz;
                if (uij_xij < 0) {
                    double h_ij = (hi + hj) * 0.5;
                    double phi_ij = h_ij * uij_xij;
                    phi_ij /= (tdist * tdist + 0.01 * h_ij * h_ij);
                    double P_ij = mi * phi_ij * (-Alpha * soundspeed + Beta * phi_ij);
                    P_ij /= (rhoi + rhoj);
                    P_ij *= 0.5;
                    v2[0] = -(P_ij)*tdwx; v2[1] = -(P_ij)*tdwy; v2[2] = -(P_ij)*tdwz;
                }
            }
        }
        sums.template add<ADV_SECOND>(v, v2, art);
        if (SCAL && (concn_solve || boussinesq_solve)) sums2.template add<1>(w, w2, true);
    }
    AdvSums a;
    a.tx = sums.sum(0); a.ty = sums.sum(1); a.tz = sums.sum(2);
    a.cx = sums.sum(3); a.cy = sums.sum(4); a.cz = sums.sum(5);
    if constexpr (SCAL) {
        a.rc = sums.sum(6); a.ct = sums.sum(7);
        a.rd = sums2.sum(0); a.temp = sums2.sum(1); a.flt = sums2.sum(2);
    }
    if (g_ == 0) advection_store(cd, i, a, con_solve, concn_solve, boussinesq_solve, cpi);
}

// MIXED (see prep_sums)
template <bool SCAL, bool REC, class Src, int W>
__device__ __forceinline__ void advection_sums(const CaseDesc& cd, int i, const NLRow row, const Src src, int g,
                                               bool con_solve, bool concn_solve, bool boussinesq_solve, AdvSums& a) {
    const KConst kc = cd.kc;
    const sph_params& pr = cd.pr;
    const PView S = cd.S;
    const Rec rec(cd);
    const int ptypei = S.p_type[i];
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    const float xf = (float)xi, yf = (float)yi, zf = (float)zi;
    const double uxi = S.ux[i], uyi = S.uy[i], uzi = S.uz[i];
    const float fux = (float)uxi, fuy = (float)uyi, fuz = (float)uzi;
    const double tempi = SCAL ? S.temp[i] : 0.0;
    const float concni = SCAL ? (float)S.concn[i] : 0.0f;
    const double hi_d = S.h[i], eli = S.eli[i];
    const float hi = (float)hi_d, mi = (float)S.m[i], rhoi = (float)S.rho[i];
    const float tmp_A = calc_tmpA<float>(kc, hi), f = dw_factor<float>(kc, hi);
    const HScale hs(kc, hi);
    const float kci = SCAL ? (float)(pr.solid_k * (ptypei == 0 || ptypei == 1000) + pr.air_k * (ptypei == 1 || ptypei == -1)) : 0.0f;
    const float visi = (float)(viscosity2(pr, ptypei) + S.vis_t[i] * S.rho[i]);
    const float ome = (float)(1 - eli);
    const bool conv = eli < 1.0, av = pr.artificial_viscosity != 0;
    const int fv = pr.fv_solve;
    const float Alpha = (float)pr.av_alpha, Beta = (float)pr.av_beta, soundspeed = (float)pr.av_c;
    // consecutive neighbours mostly share rho: the reciprocals it enters are kept
    float rho_c = NO_VALUE, yrho = 0.0f, rr = 0.0f, yrr = 0.0f, rs = 0.0f, yrs = 0.0f;
    walk_row<REC, 2, 2, W>(row, src, g, [&](unsigned e, const Pieces<2, 2>& rec_) {
        if (!(e & F_DP)) return;
        const int j = e & NB_IDX;
        float dx, dy, dz, mj, rhoj, visj;
        float dux, duy, duz;   // u_i - u_j
        double hj_d;
        int ptypej;
        if constexpr (REC) {   // (every piece is read here: see walk_row)
            const rec_f4 p = rec_.f[0], b = rec_.f[1];
            const rec_d2 u = rec_.d[0], w = rec_.d[1];
            ptypej = crec_ptype(b.w);
            dx = xf - p.x; dy = yf - p.y; dz = zf - p.z; mj = p.w;
            rhoj = b.x; hj_d = b.y; visj = b.z;
            dux = (float)(uxi - u.x); duy = (float)(uyi - u.y); duz = (float)(uzi - w.x);
            if (ptypej >= 1000) return;
        } else {
            double vis_tj, xj, yj, zj, mj_d, rhoj_d, pqj_, uxj, uyj, uzj;
            int itj_;
            rec_aux(rec, j, vis_tj, ptypej, itj_);
            if (ptypej >= 1000) return;
            rec_pos(rec, j, xj, yj, zj, mj_d, rhoj_d, pqj_);
            rec_vel(rec, j, uxj, uyj, uzj, hj_d);
            dx = (float)(xi - xj); dy = (float)(yi - yj); dz = (float)(zi - zj);
            mj = (float)mj_d; rhoj = (float)rhoj_d;
            visj = (float)(viscosity2(pr, ptypej) + vis_tj * rhoj_d);
            dux = (float)(uxi - uxj); duy = (float)(uyi - uyj); duz = (float)(uzi - uzj);
        }
        if (rhoj != rho_c) {
            rho_c = rhoj;
            yrho = recip(rhoj);
            rr = rhoi * rhoj; yrr = recip(rr);
            rs = rhoi + rhoj; yrs = recip(rs);
        }
        const Dist d = dist_of(dx * dx + dy * dy + dz * dz);
        const float tR = hs.tR(d.r), dw = kernel_dw_t<float>(kc, tmp_A, f, tR);
        const float tx = quot(dw * dx, d.r, d.y), ty = quot(dw * dy, d.r, d.y), tz = quot(dw * dz, d.r, d.y);
        if (fv == SPH_FV_CLEARY) {
            float C_v = dx * tx + dy * ty + dz * tz;
            const float vs = visi + visj;
            C_v *= quot(visi * visj, vs, recip(vs));
            C_v *= 4.0f * quot_any(mj, rr, yrr);
            C_v = quot(quot(C_v, d.r, d.y), d.r, d.y);
            a.tx += (double)(C_v * dux); a.ty += (double)(C_v * duy); a.tz += (double)(C_v * duz);
        } else if (fv == SPH_FV_MONAGHAN) {
            const float phi = (dux * dx + duy * dy + duz * dz) / (d.r * d.r + 0.01f * hi * hi);
            float P = -10.0f * phi * mj / rhoj;
            const float C_v = 2.0f * (visi * visj) / (visi + visj - 1e-20f);
            P *= C_v / rhoi;
            if (ptypei <= 0 || ptypei >= 1000 || ptypej <= 0) P = 0;
            a.tx += (double)(-P * tx); a.ty += (double)(-P * ty); a.tz += (double)(-P * tz);
        }
        if (conv) {
            const float vx = -dux, vy = -duy, vz = -duz;   // u_j - u_i
            a.cx += (double)(quot_any((fux * vx * tx + fuy * vx * ty + fuz * vx * tz) * mj, rhoj, yrho) * ome);
            a.cy += (double)(quot_any((fux * vy * tx + fuy * vy * ty + fuz * vy * tz) * mj, rhoj, yrho) * ome);
            a.cz += (double)(quot_any((fux * vz * tx + fuy * vz * ty + fuz * vz * tz) * mj, rhoj, yrho) * ome);
        }
        if (SCAL && (con_solve || concn_solve || boussinesq_solve)) {
            double tempj, concnj_d;
            if constexpr (REC) { tempj = S.temp[src.gidx(j)]; concnj_d = S.concn[src.gidx(j)]; }
            else rec_scalar(rec, j, tempj, concnj_d);
            if (conv && con_solve)
                a.ct -= (double)(2.0f * mj / rs * (float)(tempj - tempi) * (dux * tx + duy * ty + duz * tz) * ome);
            if (conv && concn_solve) {
                const float dc = (float)(concnj_d - (double)concni);
                a.rd -= (double)((fux * dc * tx + fuy * dc * ty + fuz * dc * tz) * mj / rhoj * ome);
            }
            if (con_solve) {
                const float kcj = (float)(pr.solid_k * (ptypej == 0 || ptypej == 1000) + pr.air_k * (ptypej == 1 || ptypej == -1));
                const float rhoj_temp = (ptypej == 1 || ptypej == -1) ? rhoj : (float)pr.solid_rho;
                const float mj_temp = mj * rhoj_temp / rhoj;
                float H = 4.0f * mj_temp * kcj * kci * (float)(tempi - tempj) * dw;
                H /= (d.r + 1e-10f) * rhoi * rhoj_temp * (kci + kcj);
                a.rc += (double)H;
            }
            if (concn_solve) {
                const float diff = (float)pr.diff_coef;
                float D = mi * (diff * rhoi + diff * rhoj);
                D *= (dx * tx + dy * ty + dz * tz);
                D /= (rhoi * rhoj * (d.r * d.r + 0.01f * hi * hi));
                a.rd += (double)(D * (concni - (float)concnj_d) * (float)(ptypei == ptypej));
            }
            if (boussinesq_solve) {
                const float vj = mj / rhoj, twij = kernel_w_t<float>(kc, tmp_A, tR);
                a.temp += (double)(vj * (float)tempj * twij);
                a.flt += (double)(vj * twij);
            }
        }
        if (av) {
            const float ud = dux * dx + duy * dy + duz * dz;
            if (ud < 0) {
                const float h_ij = (float)((hi_d + hj_d) * 0.5);
                const float den = d.r * d.r + 0.01f * h_ij * h_ij;
                const float phi = quot(h_ij * ud, den, recip(den));
                const float P = quot_any(mi * phi * (-Alpha * soundspeed + Beta * phi), rs, yrs) * 0.5f;
                a.tx += (double)(-P * tx); a.ty += (double)(-P * ty); a.tz += (double)(-P * tz);
            }
        }
    });
}
template <bool SCAL, class Src, int W = 1>
__device__ __forceinline__ void advection_mixed(const CaseDesc& cd, int i, const NList& nl, int li, const Src src,
                                                int g = 0) {
    const sph_params& pr = cd.pr;
    const bool con = SCAL && pr.con_solve, concn = SCAL && pr.concn_solve, bous = SCAL && pr.boussinesq_solve;
    const int ptypei = cd.S.p_type[i];
    if (cd.S.i_type[i] > 2) return;
    if (ptypei == 1000) return;
    if (ptypei <= 0) return;
    AdvSums a;
    const NLRow row = nl_row(nl, li);
    if constexpr (Src::lds) {
        advection_sums<SCAL, true, Src, W>(cd, i, row, src, g, con, concn, bous, a);
    } else {
        if (src.ok()) advection_sums<SCAL, true, Src, W>(cd, i, row, src, g, con, concn, bous, a);
        else advection_sums<SCAL, false, Src, W>(cd, i, row, src, g, con, concn, bous, a);
    }
    if constexpr (W > 1) {
        group_fold<W>(a.tx); group_fold<W>(a.ty); group_fold<W>(a.tz);
        group_fold<W>(a.cx); group_fold<W>(a.cy); group_fold<W>(a.cz);
        if (SCAL) {
            group_fold<W>(a.rc); group_fold<W>(a.rd); group_fold<W>(a.ct); group_fold<W>(a.temp); group_fold<W>(a.flt);
        }
        if (g != 0) return;
    }
    double cpi = 1.0;
    if (con)
        cpi = (double)(float)(pr.solid_cp * (ptypei == 0 || ptypei == 1000) + pr.air_cp * (ptypei == 1 || ptypei == -1));
    advection_store(cd, i, a, con, concn, bous, cpi);
}
template <bool SCAL>
__global__ void __launch_bounds__(MAX_BLOCK) k_advection_mixed(Seg sg) {
    SEG_GROUP_LIGHT(sg);
    advection_mixed<SCAL, GSrc, GROUP>(cd, i, cd.nl, i, GSrc{&cd.crec_adv, (size_t)cd.n}, g_);
}
template <bool SCAL>
__global__ void __launch_bounds__(WAVE_BLOCK) k_advection_heavy(Seg sg) {
    SEG_HEAVY(sg);
    advection_mixed<SCAL, GSrc, 64>(cd, i, cd.nl, i, GSrc{&cd.crec_adv, (size_t)cd.n}, lane_);
}
template <bool SCAL>
__global__ void __launch_bounds__(TILE_THREADS) k_advection_tile(Seg sg, int width) {
    TILE_CHUNK(sg, width, cd.crec_adv, CREC_ADV_FLOATS);
    TILE_LANES(width) {
        if (chunk_.y >= 0)
            advection_mixed<SCAL, LSrc<CREC_ADV_FLOATS>, GROUP>(cd, i, cd.tile.nl, lane_, TILE_SRC(CREC_ADV_FLOATS), g_);
        else
            advection_mixed<SCAL, GSrc, GROUP>(cd, i, cd.tile.nl, lane_,
                                                                GSrc{&cd.crec_adv, (size_t)cd.n}, g_);
    }
}

// ------------------------------------------------------------------------
// KERNEL_clc_projection, functions_TIME_ISPH.cuh:2-112 (predictor)
__global__ void __launch_bounds__(MAX_BLOCK) k_projection(Seg sg) {
    SEG_PARTICLE(sg);
    const sph_params pr = cd.pr;
    if (pr.time_type != SPH_PRE_COR) return;   // ISPH_Calc.cuh:105
    const PView S = cd.S;
    const P2View S2 = cd.S2;
    const QView Q = cd.Q;
    const double dt = cd.dt, time = cd.time;
    if (S.i_type[i] >= 3) return;
    if (S.p_type[i] >= 1000) return;
    int buffer_type = S.buffer_type[i], MOST = S.MOST_buffer[i], p_typei = S.p_type[i];
    if (p_typei == 9) {
        S2.x0[i] = S.x[i]; S2.y0[i] = S.y[i]; S2.z0[i] = S.z[i];
        S.ux[i] = 1.0; S.uy[i] = 0; S.uz[i] = 0;
        S2.ux0[i] = 1.0; S2.uy0[i] = 0; S2.uz0[i] = 0;
    } else {
        double tux0 = S.ux[i], tuy0 = S.uy[i], tuz0 = S.uz[i];
        double tuxp, tuyp, tuzp;
        if (p_typei > 0) {
            double b = (double)(buffer_type == 0 || MOST == 1);
            double tdux = Q.ftotalx[i] * b + S.fmx[i];
            double tduy = Q.ftotaly[i] * b + S.fmy[i];
            double tduz = Q.ftotalz[i] * b;
            tuxp = tux0 + tdux * (dt);
            tuyp = tuy0 + tduy * (dt);
            tuzp = tuz0 + tduz * (dt);
        } else {
            tuxp = tux0; tuyp = tuy0; tuzp = tuz0;
        }
        S.ux[i] = tuxp; S.uy[i] = tuyp; S.uz[i] = tuzp;
        S2.x0[i] = S.x[i]; S2.y0[i] = S.y[i]; S2.z0[i] = S.z[i];
        S2.ux0[i] = tux0; S2.uy0[i] = tuy0; S2.uz0[i] = tuz0;
    }
    if (time == 0) S2.rho_ref[i] = S.rho[i];
    if (pr.con_solve == 1) S2.temp0[i] = S.temp[i];
    if (pr.concn_solve == 1) {
        double tconcn = S.concn[i];
        S2.concn0[i] = tconcn;
        S.concn[i] = tconcn + Q.dconcn[i] * (dt);
    }
}

// ------------------------------------------------------------------------
// KERNEL_periodic_boundary3D, functions_BC.cuh:1015-1154 (reads the snapshot
// arrays; last match inside the first cell that has one).
__global__ void __launch_bounds__(MAX_BLOCK) k_periodic(Seg sg, int which) {
    SEG_PARTICLE(sg);
    const sph_params pr = cd.pr;
    const PView A = which ? cd.P : cd.S;
    const Grid g = cd.g;
    const double *oux = cd.snap[0], *ouy = cd.snap[1], *ouz = cd.snap[2], *opres = cd.snap[3], *otemp = cd.snap[4];
    int bt = A.buffer_type[i];
    if (bt == 0) return;
    if (A.p_type[i] >= 1000) return;
    double xi = A.x[i], yi = A.y[i], zi = A.z[i];
    double xg, yg, zg;
    if (bt == 3) { xg = xi; yg = yi + pr.L_right - pr.L_left; zg = zi; }
    else if (bt == 4) { xg = xi; yg = yi - pr.L_right + pr.L_left; zg = zi; }
    else return;
    const sph_domain& d = g.d;
    int nc = A.ncell[i];
    Cell c = query_cell(d, xg, yg, zg);
    int found = -1;
    // only cells inside the bin range of the copy_tol ball can hold a match
    // (the first such cell in window order is unchanged)
    Cell lo, hi;
    ball_bins(d, xg, yg, zg, pr.copy_tol, lo, hi);
    for (int z = max(-nc, lo.k - c.k); z <= min(nc, hi.k - c.k) && found < 0; z++)
        for (int y = max(-nc, lo.j - c.j); y <= min(nc, hi.j - c.j) && found < 0; y++)
            for (int x = max(-nc, lo.i - c.i); x <= min(nc, hi.i - c.i) && found < 0; x++) {
                if (!cell_ok(d, c.i + x, c.j + y, c.k + z)) continue;
                int cell = (c.i + x) + d.NI * (c.j + y) + d.NI * d.NJ * (c.k + z);
                int s = g.gstr[cell];
                if (s == -1) continue;
                int e = g.gend[cell];
                for (int j = s; j < e; j++) {
                    double tdist = dist3<double>(xg, yg, zg, A.x[j], A.y[j], A.z[j]) - 1e-20;
                    if (tdist < pr.copy_tol) found = j;
                }
            }
    if (found >= 0) {
        A.ux[i] = oux[found]; A.uy[i] = ouy[found]; A.uz[i] = ouz[found];
        A.pres[i] = opres[found]; A.temp[i] = otemp[found];
    } else {
        A.ux[i] = 0; A.uy[i] = 0; A.uz[i] = 0; A.pres[i] = 0; A.temp[i] = 0;
    }
}

// ------------------------------------------------------------------------
// KERNEL_freeslip_boundary3D, functions_BC.cuh:1156-1271
constexpr int FS_SUMS = 6;
__global__ void __launch_bounds__(WAVE_BLOCK) k_freeslip(Seg sg, int which) {
    __shared__ double lds[WAVE_BLOCK / 64][ord_doubles(FS_SUMS)];
    SEG_BOUNDARY(sg);
    const KConst kc = cd.kc;
    const PView A = which ? cd.P : cd.S;
    if (A.p_type[i] != -1) return;
    const double hi = A.h[i], tmp_A = calc_tmpA<double>(kc, hi);
    const double xg = A.x[i], yg = A.y[i], zg = A.z[i];
    OrderedSums<FS_SUMS, BLANES> sums(lds[threadIdx.x >> 6]);
    const NLRow row = nl_row(cd.nl, i);
    for (int k = lane; k - lane < row.cnt; k += BLANES) {
        const unsigned e = k < row.cnt ? NB_AT(row, k) : 0u;
        const int j = e & NB_IDX;
        double v[FS_SUMS] = {};
        // fluid neighbours only (the reference weights the others by an
        // exact 0, which leaves the sums unchanged)
        if ((e & F_HM) && A.p_type[j] == 1) {
            const double dx = xg - A.x[j], dy = yg - A.y[j], dz = zg - A.z[j];
            const double tdist = sqrt(dx * dx + dy * dy + dz * dz) - 1e-20;
            const double mj = A.m[j], rhoj = A.rho[j];
            const double twij = kernel_w<double>(kc, tmp_A, hi, tdist);
            v[0] = A.ux[j] * (mj / rhoj) * twij;
            v[1] = A.uy[j] * (mj / rhoj) * twij;
            v[2] = A.uz[j] * (mj / rhoj) * twij;
            v[3] = A.pres[j] * (mj / rhoj) * twij;
            v[4] = A.temp[j] * (mj / rhoj) * twij;
            v[5] = (mj / rhoj) * twij;
        }
        sums.add(v);
    }
    double t[FS_SUMS];
    for (int a = 0; a < FS_SUMS; a++) t[a] = sums.sum(a);
    if (lane != 0) return;
    if (t[5] > 1e-5) {
        A.ux[i] = t[0] / t[5]; A.uy[i] = t[1] / t[5]; A.uz[i] = t[2] / t[5];
        A.pres[i] = t[3] / t[5]; A.temp[i] = t[4] / t[5];
    }
}

// The same sums in MIXED (see k_boundary3d_mixed)
__global__ void __launch_bounds__(WAVE_BLOCK) k_freeslip_mixed(Seg sg, int which) {
    SEG_BOUNDARY(sg);
    const PView A = which ? cd.P : cd.S;
    if (A.p_type[i] != -1) return;
    const KConst kc = cd.kc;
    const NList nl = cd.nl;
    const float hi = (float)A.h[i], tmp_A = calc_tmpA<float>(kc, hi);
    const HScale hs(kc, hi);
    float rho_c = NO_VALUE, yrho = 0.0f;
    double xg = A.x[i], yg = A.y[i], zg = A.z[i];
    double t[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const NLRow row = nl_row(nl, i);
    for (int k = lane; k < row.cnt; k += BLANES) {
        unsigned e = NB_AT(row, k);
        if (!(e & F_HM)) continue;
        int j = e & NB_IDX;
        if (A.p_type[j] != 1) continue;
        float dx = (float)(xg - A.x[j]), dy = (float)(yg - A.y[j]), dz = (float)(zg - A.z[j]);
        const float rhoj = (float)A.rho[j];
        if (rhoj != rho_c) { rho_c = rhoj; yrho = recip(rhoj); }
        const float vj = quot_any((float)A.m[j], rhoj, yrho);
        const float w = kernel_w_t<float>(kc, tmp_A, hs.tR(dist_of(dx * dx + dy * dy + dz * dz).r));
        t[0] += (double)((float)A.ux[j] * vj * w);
        t[1] += (double)((float)A.uy[j] * vj * w);
        t[2] += (double)((float)A.uz[j] * vj * w);
        t[3] += (double)((float)A.pres[j] * vj * w);
        t[4] += (double)((float)A.temp[j] * vj * w);
        t[5] += (double)(vj * w);
    }
    for (double& v : t) group_fold<BLANES>(v);
    if (lane != 0) return;
    if (t[5] > 1e-5) {
        A.ux[i] = t[0] / t[5]; A.uy[i] = t[1] / t[5]; A.uz[i] = t[2] / t[5];
        A.pres[i] = t[3] / t[5]; A.temp[i] = t[4] / t[5];
    }
}

// ------------------------------------------------------------------------
// KERNEL_donothing_buffer3D, functions_BC.cuh:673-761 (snapshot reads)
__global__ void __launch_bounds__(MAX_BLOCK) k_outlet(Seg sg, int which) {
    SEG_PARTICLE(sg);
    const sph_params pr = cd.pr;
    const PView A = which ? cd.P : cd.S;
    const Grid g = cd.g;
    const double *oux = cd.snap[0], *ouy = cd.snap[1], *ouz = cd.snap[2], *opres = cd.snap[3], *otemp = cd.snap[4];
    if (A.buffer_type[i] != 2) return;
    const sph_domain& d = g.d;
    double xi = A.x[i], yi = A.y[i], zi = A.z[i];
    Cell c = query_cell(d, xi, yi, zi);
    int nc = 2 * A.ncell[i];
    double xg = pr.L3 - pr.outlet_copy_dx;
    int found = -1;
    // A match lies within copy_tol of (xg, yi, zi); binning is monotone, so
    // only window cells inside the bin range of that ball can hold one.
    // Skipping the others leaves the last match in window order unchanged.
    Cell lo, hi;
    ball_bins(d, xg, yi, zi, pr.copy_tol, lo, hi);
    for (int z = max(-nc, lo.k - c.k); z <= min(nc, hi.k - c.k); z++)
        for (int y = max(-nc, lo.j - c.j); y <= min(nc, hi.j - c.j); y++)
            for (int x = max(-nc, lo.i - c.i); x <= min(nc, hi.i - c.i); x++) {
                if (!cell_ok(d, c.i + x, c.j + y, c.k + z)) continue;
                int cell = (c.i + x) + d.NI * (c.j + y) + d.NI * d.NJ * (c.k + z);
                int s = g.gstr[cell];
                if (s == -1) continue;
                int e = g.gend[cell];
                for (int j = s; j < e; j++) {
                    double tdist = dist3<double>(xg, yi, zi, A.x[j], A.y[j], A.z[j]) - 1e-20;
                    if (A.p_type[j] < 1000 && tdist < pr.copy_tol) found = j;
                }
            }
    if (found >= 0) {
        A.pres[i] = opres[found]; A.ux[i] = oux[found]; A.uy[i] = ouy[found]; A.uz[i] = ouz[found];
        A.temp[i] = otemp[found];
    } else {
        A.pres[i] = 0; A.ux[i] = 0; A.uy[i] = 0; A.uz[i] = 0; A.temp[i] = 0;
    }
}

// ------------------------------------------------------------------------
// KERNEL_pressureforce3D, functions_PPE.cuh:482-647
__device__ __forceinline__ bool pressure_row(const PView& S, int i) {
    return S.i_type[i] <= 2 && S.p_type[i] < 1000 && S.p_type[i] > 0 && S.buffer_type[i] == 0;
}
constexpr int PF_SUMS = 3;
__global__ void __launch_bounds__(MAX_BLOCK) k_pressure_force(Seg sg) {
    ORDERED_LDS(PF_SUMS, 0);
    SEG_GROUP_LIGHT(sg);
    const KConst kc = cd.kc;
    const PView S = cd.S;
    const QView Q = cd.Q;
    if (!pressure_row(S, i)) return;
    const bool on = cd.pr.fp_solve != 0;
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    const double hi = S.h[i];
    const double pi = S.pres[i] - S.pres0[i], rhoi = S.rho[i];
    // the pair's kernel normalisation and derivative factor depend only on
    // h_ij: kept while a lane's consecutive pairs share it
    double h_c = -1, A_c = 0, f_c = 0;
    OrderedSums<PF_SUMS, GROUP> sums(wlds_);
    const NLRow row = nl_row(cd.nl, i);
    for (int k = g_; k - g_ < row.cnt && on; k += GROUP) {
        const unsigned e = k < row.cnt ? NB_AT(row, k) : 0u;
        const int j = e & NB_IDX;
        const bool pair = (e & F_DM) && S.p_type[j] < 1000;
        if (!__any(pair)) continue;
        double v[PF_SUMS] = {};
        if (pair) {
            double hj, pj, xj, yj, zj, mj, rhoj;
            rec_pos(Rec(cd), j, xj, yj, zj, mj, rhoj, pj);
            hj = Rec(cd).piece(j, 4).y;
            const double dx = xi - xj, dy = yi - yj, dz = zi - zj;
            const double tdist = sqrt(dx * dx + dy * dy + dz * dz) - 1e-20;
            const double hij = 0.5 * (hi + hj);
            if (hij != h_c) { h_c = hij; A_c = calc_tmpA<double>(kc, hij); f_c = dw_factor<double>(kc, hij); }
            const double tdwij = kernel_dw_f<double>(kc, A_c, hij, f_c, tdist);
            const double Pb = 0.0;
            const double C_p = -2.0 * mj / (rhoi * rhoj) * ((pi + Pb) * rhoj + (pj + Pb) * rhoi) / (rhoi + rhoj);
            v[0] = C_p * (tdwij * dx / tdist);
            v[1] = C_p * (tdwij * dy / tdist);
            v[2] = C_p * (tdwij * dz / tdist);
        }
        sums.add(v);
    }
    const double tx = sums.sum(0), ty = sums.sum(1), tz = sums.sum(2);
    if (g_ == 0) { Q.fpx[i] = tx; Q.fpy[i] = ty; Q.fpz[i] = tz; }
}

// MIXED (see prep_sums)
template <bool REC, class Src, int W>
__device__ __forceinline__ void pressure_sums(const CaseDesc& cd, int i, const NLRow row, const Src src, int g,
                                              double& tmpx, double& tmpy, double& tmpz) {
    const KConst kc = cd.kc;
    const PView S = cd.S;
    const Rec rec(cd);
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i], hi_d = S.h[i];
    const float xf = (float)xi, yf = (float)yi, zf = (float)zi;
    const float pi = (float)(S.pres[i] - S.pres0[i]), rhoi = (float)S.rho[i];
    // the pair's kernel normalisation and derivative factor depend only on
    // h_ij, its density terms on rho_j: kept while consecutive pairs share them
    float h_c = -1.0f, A_c = 0.0f, f_c = 0.0f;
    HScale hs(kc, 1.0f);
    float rho_c = NO_VALUE, rr = 0.0f, yrr = 0.0f, rs = 0.0f, yrs = 0.0f;
    walk_row<REC, 2, 0, W>(row, src, g, [&](unsigned e, const Pieces<2, 0>& rec_) {
        if (!(e & F_DM)) return;
        const int j = e & NB_IDX;
        float dx, dy, dz, mj, rhoj, pj;
        double hj;
        if constexpr (REC) {
            const rec_f4 p = rec_.f[0], b = rec_.f[1];
            if (__float_as_int(b.w) >= 1000) return;
            dx = xf - p.x; dy = yf - p.y; dz = zf - p.z; mj = p.w;
            rhoj = b.x; pj = b.y; hj = b.z;
        } else {
            if (S.p_type[j] >= 1000) return;
            double xj, yj, zj, mj_d, rhoj_d, pqj;
            rec_pos(rec, j, xj, yj, zj, mj_d, rhoj_d, pqj);
            hj = rec.piece(j, 4).y;
            dx = (float)(xi - xj); dy = (float)(yi - yj); dz = (float)(zi - zj);
            mj = (float)mj_d; rhoj = (float)rhoj_d; pj = (float)pqj;
        }
        const float hij = (float)(0.5 * (hi_d + hj));
        if (hij != h_c) {
            h_c = hij;
            A_c = calc_tmpA<float>(kc, hij);
            f_c = dw_factor<float>(kc, hij);
            hs = HScale(kc, hij);
        }
        if (rhoj != rho_c) {
            rho_c = rhoj;
            rr = rhoi * rhoj; yrr = recip(rr);
            rs = rhoi + rhoj; yrs = recip(rs);
        }
        const Dist d = dist_of(dx * dx + dy * dy + dz * dz);
        const float dw = kernel_dw_t<float>(kc, A_c, f_c, hs.tR(d.r));
        const float tx = quot(dw * dx, d.r, d.y), ty = quot(dw * dy, d.r, d.y), tz = quot(dw * dz, d.r, d.y);
        const float C_p = quot_any(quot_any(-2.0f * mj, rr, yrr) * (pi * rhoj + pj * rhoi), rs, yrs);
        tmpx += (double)(C_p * tx); tmpy += (double)(C_p * ty); tmpz += (double)(C_p * tz);
    });
}
template <class Src, int W = 1>
__device__ __forceinline__ void pressure_force_mixed(const CaseDesc& cd, int i, const NList& nl, int li,
                                                     const Src src, int g = 0) {
    if (!pressure_row(cd.S, i)) return;
    double tx = 0, ty = 0, tz = 0;
    const NLRow row = nl_row(nl, li);
    if (cd.pr.fp_solve) {
        if constexpr (Src::lds) {
            pressure_sums<true, Src, W>(cd, i, row, src, g, tx, ty, tz);
        } else {
            if (src.ok()) pressure_sums<true, Src, W>(cd, i, row, src, g, tx, ty, tz);
            else pressure_sums<false, Src, W>(cd, i, row, src, g, tx, ty, tz);
        }
    }
    if constexpr (W > 1) {
        group_fold<W>(tx); group_fold<W>(ty); group_fold<W>(tz);
        if (g != 0) return;
    }
    const QView Q = cd.Q;
    Q.fpx[i] = tx; Q.fpy[i] = ty; Q.fpz[i] = tz;
}
__global__ void __launch_bounds__(MAX_BLOCK) k_pressure_force_mixed(Seg sg) {
    SEG_GROUP_LIGHT(sg);
    pressure_force_mixed<GSrc, GROUP>(cd, i, cd.nl, i, GSrc{&cd.crec, (size_t)cd.n}, g_);
}
__global__ void __launch_bounds__(WAVE_BLOCK) k_pressure_force_heavy(Seg sg) {
    SEG_HEAVY(sg);
    pressure_force_mixed<GSrc, 64>(cd, i, cd.nl, i, GSrc{&cd.crec, (size_t)cd.n}, lane_);
}
__global__ void __launch_bounds__(TILE_THREADS) k_pressure_force_tile(Seg sg, int width) {
    TILE_CHUNK(sg, width, cd.crec, CREC_FLOATS);
    TILE_LANES(width) {
        if (chunk_.y >= 0) pressure_force_mixed<LSrc<CREC_FLOATS>, GROUP>(cd, i, cd.tile.nl, lane_, TILE_SRC(CREC_FLOATS), g_);
        else pressure_force_mixed<GSrc, GROUP>(cd, i, cd.tile.nl, lane_, GSrc{&cd.crec, (size_t)cd.n}, g_);
    }
}

// ------------------------------------------------------------------------
// IBM_force_interpolation3D, functions_IBM.cuh:342-490
// the force from the interpolated velocity's sums
__device__ __forceinline__ void ibm_force_store(const CaseDesc& cd, int i, const double (&t)[4]) {
    const sph_params& pr = cd.pr;
    const PView S = cd.S;
    const QView Q = cd.Q;
    const double dt = cd.dt, zi = S.z[i], filt = t[3];
    S.concentration[i] = filt;
    double ufx = t[0] / (filt + 1e-10), ufy = t[1] / (filt + 1e-10), ufz = t[2] / (filt + 1e-10);
    double nx = Q.nx[i], ny = Q.ny[i], nz = Q.nz[i];
    double nmag = sqrt(nx * nx + ny * ny + nz * nz) + 1e-20;
    nx = nx / nmag; ny = ny / nmag; nz = nz / nmag;
    double un = ufx * nx + ufy * ny + ufz * nz;
    double utx = ufx - un * nx, uty = ufy - un * ny, utz = ufz - un * nz;
    double Ubtx = pr.ibm_ut_factor * interp_ux_caseH(zi, 1.0);
    double Ubty = 0.0, Ubtz = 0.0;
    double beta_t = 1.0;
    double corrx = (-un) * nx + beta_t * (Ubtx - utx);
    double corry = (-un) * ny + beta_t * (Ubty - uty);
    double corrz = (-un) * nz + beta_t * (Ubtz - utz);
    S.fbx[i] = pr.rho_air * corrx / dt;
    S.fby[i] = pr.rho_air * corry / dt;
    S.fbz[i] = pr.rho_air * corrz / dt;
}
__global__ void __launch_bounds__(WAVE_BLOCK) k_ibm_force(Seg sg) {
    __shared__ double lds[WAVE_BLOCK / 64][ord_doubles(4)];
    SEG_BOUNDARY(sg);
    const KConst kc = cd.kc;
    const PView S = cd.S;
    if (S.p_type[i] < 1000) return;
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    const double tmp_h = 0.5 * S.h[i], tmp_A = calc_tmpA<double>(kc, tmp_h);
    OrderedSums<4, BLANES> sums(lds[threadIdx.x >> 6]);
    const NLRow row = nl_row(cd.nl, i);
    for (int k = lane; k - lane < row.cnt; k += BLANES) {
        const unsigned e = k < row.cnt ? NB_AT(row, k) : 0u;
        const int j = e & NB_IDX;
        double v[4] = {};
        if ((e & F_BH) && S.i_type[j] != 4 && S.p_type[j] == 1) {
            const double dx = xi - S.x[j], dy = yi - S.y[j], dz = zi - S.z[j];
            const double tdist = sqrt(dx * dx + dy * dy + dz * dz) + 1e-20;
            const double twij = kernel_w<double>(kc, tmp_A, tmp_h, tdist);
            const double tmprho = S.m[j] / S.rho[j];
            v[0] = S.ux[j] * tmprho * twij;
            v[1] = S.uy[j] * tmprho * twij;
            v[2] = S.uz[j] * tmprho * twij;
            v[3] = tmprho * twij;
        }
        sums.add(v);
    }
    double t[4];
    for (int a = 0; a < 4; a++) t[a] = sums.sum(a);
    if (lane == 0) ibm_force_store(cd, i, t);
}

// The marker force in MIXED (see k_boundary3d_mixed)
__global__ void __launch_bounds__(WAVE_BLOCK) k_ibm_force_mixed(Seg sg) {
    SEG_BOUNDARY(sg);
    const PView S = cd.S;
    if (S.p_type[i] < 1000) return;
    const KConst kc = cd.kc;
    const NList nl = cd.nl;
    double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    const float tmp_h = (float)(0.5 * S.h[i]), tmp_A = calc_tmpA<float>(kc, tmp_h);
    const HScale hs(kc, tmp_h);
    double t[4] = {0.0, 0.0, 0.0, 0.0};
    const NLRow row = nl_row(nl, i);
    for (int k = lane; k < row.cnt; k += BLANES) {
        unsigned e = NB_AT(row, k);
        if (!(e & F_BH)) continue;
        int j = e & NB_IDX;
        if (S.i_type[j] == 4 || S.p_type[j] != 1) continue;
        float dx = (float)(xi - S.x[j]), dy = (float)(yi - S.y[j]), dz = (float)(zi - S.z[j]);
        const float w = kernel_w_t<float>(kc, tmp_A, hs.tR(dist_of(dx * dx + dy * dy + dz * dz).r));
        const float tmprho = (float)S.m[j] / (float)S.rho[j];
        t[0] += (double)((float)S.ux[j] * tmprho * w);
        t[1] += (double)((float)S.uy[j] * tmprho * w);
        t[2] += (double)((float)S.uz[j] * tmprho * w);
        t[3] += (double)(tmprho * w);
    }
    for (double& v : t) group_fold<BLANES>(v);
    if (lane == 0) ibm_force_store(cd, i, t);
}

// IBM_spreading_interpolation3D, functions_IBM.cuh:492-613
__device__ __forceinline__ void ibm_spread_store(const PView& S, int i, double fb_x, double fb_y, double fb_z,
                                                 double filt) {
    if (filt < 1e-12) {
        S.fbx[i] = 0.0; S.fby[i] = 0.0; S.fbz[i] = 0.0; S.concentration[i] = 0.0;
        return;
    }
    S.fbx[i] = fb_x / (filt + 1e-10);
    S.fby[i] = fb_y / (filt + 1e-10);
    S.fbz[i] = fb_z / (filt + 1e-10);
    S.concentration[i] = filt;
}
__global__ void __launch_bounds__(MAX_BLOCK) k_ibm_spread(Seg sg) {
    ORDERED_LDS(4, 0);
    SEG_GROUP(sg);
    const KConst kc = cd.kc;
    const PView S = cd.S;
    if (S.p_type[i] != 1) return;
    if (S.buffer_type[i] == 2) return;
    if (cd.ibm_near && !cd.ibm_near[i]) {   // no marker in the list: what the sums below give
        if (g_ == 0) ibm_spread_store(S, i, 0.0, 0.0, 0.0, 0.0);
        return;
    }
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    const double tmp_h = 0.5 * S.h[i], tmp_A = calc_tmpA<double>(kc, tmp_h);
    OrderedSums<4, GROUP> sums(wlds_);
    const NLRow row = nl_row(cd.nl, i);
    for (int k = g_; k - g_ < row.cnt; k += GROUP) {
        const unsigned e = k < row.cnt ? NB_AT(row, k) : 0u;
        const int j = e & NB_IDX;
        const bool pair = (e & F_BH) && S.i_type[j] != 4 && S.p_type[j] == 1000;
        if (!__any(pair)) continue;
        double v[4] = {};
        if (pair) {
            const double dx = xi - S.x[j], dy = yi - S.y[j], dz = zi - S.z[j];
            const double tdist = sqrt(dx * dx + dy * dy + dz * dz) + 1e-20;
            const double twij = kernel_w<double>(kc, tmp_A, tmp_h, tdist);
            const double tmprho = S.m[j] / S.rho[j];
            v[0] = S.fbx[j] * twij * tmprho;
            v[1] = S.fby[j] * twij * tmprho;
            v[2] = S.fbz[j] * twij * tmprho;
            v[3] = tmprho * twij;
        }
        sums.add(v);
    }
    const double fx = sums.sum(0), fy = sums.sum(1), fz = sums.sum(2), filt = sums.sum(3);
    if (g_ == 0) ibm_spread_store(S, i, fx, fy, fz, filt);
}
// MIXED: GROUP lanes a particle, the pair arithmetic in float, the sums in
// double
__global__ void __launch_bounds__(MAX_BLOCK) k_ibm_spread_mixed(Seg sg) {
    SEG_GROUP(sg);
    const KConst kc = cd.kc;
    const PView S = cd.S;
    if (S.p_type[i] != 1) return;
    if (S.buffer_type[i] == 2) return;
    if (cd.ibm_near && !cd.ibm_near[i]) {   // no marker in the list: what the sums below give
        if (g_ == 0) ibm_spread_store(S, i, 0.0, 0.0, 0.0, 0.0);
        return;
    }
    const double xi = S.x[i], yi = S.y[i], zi = S.z[i];
    const float tmp_h = (float)(0.5 * S.h[i]), tmp_A = calc_tmpA<float>(kc, tmp_h);
    const HScale hs(kc, tmp_h);
    double filt = 0, fb_x = 0, fb_y = 0, fb_z = 0;
    const NLRow row = nl_row(cd.nl, i);
    for (int k = g_; k < row.cnt; k += GROUP) {
        const unsigned e = NB_AT(row, k);
        if (!(e & F_BH)) continue;
        const int j = e & NB_IDX;
        if (S.i_type[j] == 4 || S.p_type[j] != 1000) continue;
        const float dx = (float)(xi - S.x[j]), dy = (float)(yi - S.y[j]), dz = (float)(zi - S.z[j]);
        const float w = kernel_w_t<float>(kc, tmp_A, hs.tR(dist_of(dx * dx + dy * dy + dz * dz).r));
        const float tmprho = (float)S.m[j] / (float)S.rho[j];
        fb_x += (double)((float)S.fbx[j] * w * tmprho);
        fb_y += (double)((float)S.fby[j] * w * tmprho);
        fb_z += (double)((float)S.fbz[j] * w * tmprho);
        filt += (double)(tmprho * w);
    }
    group_fold<GROUP>(fb_x); group_fold<GROUP>(fb_y); group_fold<GROUP>(fb_z); group_fold<GROUP>(filt);
    if (g_ == 0) ibm_spread_store(S, i, fb_x, fb_y, fb_z, filt);
}

// ------------------------------------------------------------------------
// KERNEL_time_update_projection, functions_TIME_ISPH.cuh:115-296 (corrector)
// and IBM_corrector, functions_IBM.cuh:615-725 (only its copies are live).
__global__ void __launch_bounds__(MAX_BLOCK) k_time_update(Seg sg) {
    SEG_PARTICLE(sg);
    const sph_params pr = cd.pr;
    const PView S = cd.S, P = cd.P;
    const P2View S2 = cd.S2, P2 = cd.P2;
    const QView Q = cd.Q;
    const double dt = cd.dt;
    const int count = cd.count;
    if (S.p_type[i] >= 1000) {   // IBM_corrector (no i_type filter there)
        P.fbx[i] = S.fbx[i]; P.fby[i] = S.fby[i]; P.fbz[i] = S.fbz[i];
        P.concentration[i] = S.concentration[i]; P.vol[i] = S.vol[i]; P.pres[i] = S.pres[i];
        return;
    }
    if (S.i_type[i] >= 3) return;
    int buffer_type = S.buffer_type[i], p_type_i = S.p_type[i];
    if (p_type_i == 9) {
        P.ux[i] = S.ux[i]; P.uy[i] = S.uy[i]; P.uz[i] = S.uz[i];
    } else {
        double tux0, tuy0, tuz0, dux_dt, duy_dt, duz_dt;
        if (p_type_i > 0) {
            tux0 = S.ux[i]; tuy0 = S.uy[i]; tuz0 = S.uz[i];
            if (buffer_type == 1 || buffer_type == -1) { tux0 = S2.ux0[i]; tuy0 = S2.uy0[i]; tuz0 = S2.uz0[i]; }
            double b = (double)(buffer_type == 0);
            dux_dt = Q.fpx[i] * b + S.fbx[i] / S.rho[i] + S.fmx[i];
            duy_dt = Q.fpy[i] * b + S.fby[i] / S.rho[i] + S.fmy[i];
            duz_dt = Q.fpz[i] * b + S.fbz[i] / S.rho[i];
        } else {
            tux0 = S2.ux0[i]; tuy0 = S2.uy0[i]; tuz0 = S2.uz0[i];
            dux_dt = duy_dt = duz_dt = 0.0;
        }
        double uxc = tux0 + dux_dt * (dt), uyc = tuy0 + duy_dt * (dt), uzc = tuz0 + duz_dt * (dt);
        if ((uxc * uxc + uyc * uyc + uzc * uzc) >= pr.u_limit * pr.u_limit) { uxc = tux0; uyc = tuy0; uzc = tuz0; }
        P.ux[i] = uxc; P.uy[i] = uyc; P.uz[i] = uzc;
        if (cd.xnew[0]) {
            // functions_TIME_ISPH.cuh:193-195 (computed there, written here)
            const double mv = (double)(p_type_i > 0) * S.eli[i];
            cd.xnew[0][i] = S.x[i] + (S2.ux0[i] + uxc) / 2.0 * (dt) * mv;
            cd.xnew[1][i] = S.y[i] + (S2.uy0[i] + uyc) / 2.0 * (dt) * mv;
            cd.xnew[2][i] = S.z[i] + (S2.uz0[i] + uzc) / 2.0 * (dt) * mv;
        }
    }
    if (pr.con_solve == 1) P.temp[i] = S2.temp0[i] + Q.dtemp[i] * dt * (buffer_type == 0);
    else { P.enthalpy[i] = S.enthalpy[i]; P.temp[i] = S.temp[i]; }
    if (pr.concn_solve == 1) {
        double cc = S2.concn0[i] + Q.dconcn[i] * dt;
        P.concn[i] = cc < 0.0 ? 0.0 : cc;
    } else P.concn[i] = S.concn[i];
    P.pres[i] = S.pres[i]; P.flt_s[i] = S.flt_s[i];
    P.k_turb[i] = S.k_turb[i]; P.e_turb[i] = S.e_turb[i];
    P2.rho_ref[i] = S2.rho_ref[i]; P.vis_t[i] = S.vis_t[i];
    P.fbx[i] = S.fbx[i]; P.fby[i] = S.fby[i]; P.fbz[i] = S.fbz[i];
    P.fmx[i] = S.fmx[i]; P.fmy[i] = S.fmy[i]; P.hmz[i] = S.hmz[i];
    P.float1[i] = S.float1[i]; P.float2[i] = S.float2[i]; P.float3[i] = S.float3[i];
    P.concentration[i] = S.concentration[i];
    if (P.source[i] == 1) P.concn[i] += 0.5 * dt;
    if (P.p_type[i] == 0) P.temp[i] = wall_temperature(pr, dt, count);
}

// ------------------------------------------------------------------------
// kernel_copy_max + 3 x DeviceReduce::Max, functions_OUTPUT.cuh:19-33
__device__ __forceinline__ unsigned f2ord(float f) {
    unsigned u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f(unsigned u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}
__global__ void __launch_bounds__(BLOCK) k_stats(int n, PView P, P2View S2, QView Q, unsigned* out) {
    __shared__ unsigned s[3][BLOCK];
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    float a = 0, b = 0, c = 0;
    if (i < n && !(P.p_type[i] == 0 || P.i_type[i] >= 2)) {
        a = (float)sqrt(P.ux[i] * P.ux[i] + P.uy[i] * P.uy[i] + P.uz[i] * P.uz[i]);
        b = (float)((P.rho[i] - S2.rho_ref[i]) / S2.rho_ref[i] * 100.0);
        c = (float)Q.ftotal[i];
    }
    unsigned ua = i < n ? f2ord(a) : 0u, ub = i < n ? f2ord(b) : 0u, uc = i < n ? f2ord(c) : 0u;
    s[0][threadIdx.x] = ua; s[1][threadIdx.x] = ub; s[2][threadIdx.x] = uc;
    __syncthreads();
    for (int off = BLOCK / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off)
            for (int q = 0; q < 3; q++) s[q][threadIdx.x] = max(s[q][threadIdx.x], s[q][threadIdx.x + off]);
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int q = 0; q < 3; q++) atomicMax(&out[q], s[q][0]);
}
__global__ void k_stats_final(const unsigned* in, float* out) {
    if (threadIdx.x < 3) out[threadIdx.x] = ord2f(in[threadIdx.x]);
}

// ========================================================================
// Host orchestration: every launch covers all cases of the engine's step.
// Per-case switches (noslip_bc, time_type, the count==0 Neumann call) are
// tested inside the kernels, so one launch sequence serves any mix.
// ========================================================================

// launches over the particles of every case
// a boundary pass with `lanes` lanes per boundary particle of each case
#define BOUNDL(name, kern, ...) BOUNDW(name, BLANES, kern, ##__VA_ARGS__)
#define BOUNDW(name, lanes, kern, ...)                                                                        \
    do {                                                                                            \
        Shape sh_;                                                                                  \
        SPH_TRY(shape(e, 3, WAVE_BLOCK * (64 / (lanes)), &sh_));                                                     \
        if (sh_.grid > 0) {                                                                         \
            SPH_TRY(prof_begin(e, name, 0.0));                                                      \
            hipLaunchKernelGGL(kern, dim3(sh_.grid), dim3(WAVE_BLOCK), 0, e.st, Seg{e.d_desc, sh_.tab}, ##__VA_ARGS__); \
            SPH_TRY(launch_check(&e, name));                                                        \
            SPH_TRY(prof_end(e));                                                                   \
        }                                                                                           \
    } while (0)
// the heavy-list share of a MIXED record pass: a wave per such particle
#define HEAVYL(name, kern, ...)                                                                       \
    do {                                                                                            \
        Shape sh_;                                                                                  \
        SPH_TRY(shape(e, 5, WAVE_BLOCK, &sh_));                                                     \
        if (sh_.grid > 0) {                                                                         \
            SPH_TRY(prof_begin(e, name, 0.0));                                                      \
            hipLaunchKernelGGL(kern, dim3(sh_.grid), dim3(WAVE_BLOCK), 0, e.st, Seg{e.d_desc, sh_.tab}, ##__VA_ARGS__); \
            SPH_TRY(launch_check(&e, name));                                                        \
            SPH_TRY(prof_end(e));                                                                   \
        }                                                                                           \
    } while (0)
// the cell-tile variant of a record pass: a workgroup per chunk, the halo
// records (recf floats each) in dynamic LDS
#define TILEL(name, kern, recf)                                                                      \
    do {                                                                                            \
        Shape sh_;                                                                                  \
        SPH_TRY(shape(e, 4, e.tile_lanes, &sh_));                                                   \
        if (sh_.grid > 0) {                                                                         \
            const size_t lds_ = tile_lds_bytes(e, (recf));                                          \
            SPH_TRY(tile_lds_allow(e, (const void*)(kern), lds_));                                  \
            SPH_TRY(prof_begin(e, name, 0.0));                                                      \
            hipLaunchKernelGGL(kern, dim3(sh_.grid), dim3(TILE_THREADS), lds_, e.st, Seg{e.d_desc, sh_.tab}, e.tile_lanes); \
            SPH_TRY(launch_check(&e, name));                                                        \
            SPH_TRY(prof_end(e));                                                                   \
        }                                                                                           \
    } while (0)
// GROUP lanes a particle, at the workgroup size the autotuner picked for this
// batch size (SEGO: FP64, with the LDS of nd doubles a wave for ordered sums)
#define SEGG(name, kid, kern, ...) SEGO(name, kid, 0, kern, ##__VA_ARGS__)
#define SEGO(name, kid, nd, kern, ...)                                                                   \
    do {                                                                                            \
        const int blk_ = tuned_block(e, (kid));                                                     \
        Shape sh_;                                                                                  \
        SPH_TRY(shape(e, 0, blk_ / GROUP, &sh_));                                                   \
        if (sh_.grid > 0) {                                                                         \
            SPH_TRY(prof_begin(e, name, 0.0));                                                      \
            SPH_TRY(tune_begin(e, (kid), blk_));                                                    \
            hipLaunchKernelGGL(kern, dim3(sh_.grid), dim3(blk_), (size_t)(blk_ / 64) * (nd) * sizeof(double), e.st, Seg{e.d_desc, sh_.tab}, ##__VA_ARGS__); \
            SPH_TRY(launch_check(&e, name));                                                        \
            SPH_TRY(tune_end(e));                                                                   \
            SPH_TRY(prof_end(e));                                                                   \
        }                                                                                           \
    } while (0)
#define SEGL(name, kern, ...)                                                                        \
    do {                                                                                            \
        Shape sh_;                                                                                  \
        SPH_TRY(shape(e, 0, BLOCK, &sh_));                                                          \
        if (sh_.grid > 0) {                                                                         \
            SPH_TRY(prof_begin(e, name, 0.0));                                                      \
            hipLaunchKernelGGL(kern, dim3(sh_.grid), dim3(BLOCK), 0, e.st, Seg{e.d_desc, sh_.tab}, ##__VA_ARGS__); \
            SPH_TRY(launch_check(&e, name));                                                        \
            SPH_TRY(prof_end(e));                                                                   \
        }                                                                                           \
    } while (0)

static bool mixed_of(const Eng& e) { return e.cs[0]->prm.precision == SPH_MIXED; }

// which: 0 = step working copy (SP1), 1 = persistent state (P1)
// Neumann pairs of the case's boundary particles for its current search,
// in the precision of its steps.
// 1 for a particle whose spreading list (the F_BH entries) holds an IB
// marker (p_type 1000): a superset of the particles the spreading sums
// reach, whatever the types of i and the markers' i_type become in the step
// (GROUP lanes a particle)
__global__ void __launch_bounds__(BLOCK) k_ibm_near(int n, PView S, NList nl, unsigned char* out) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x, i = t / GROUP, g = t % GROUP;
    if (i >= n) return;
    const int gbit = (int)(threadIdx.x & 63) & ~(GROUP - 1);
    bool hit = false;
    const NLRow row = nl_row(nl, i);
    for (int k0 = 0; k0 < row.cnt && !hit; k0 += GROUP) {
        const unsigned e = k0 + g < row.cnt ? NB_AT(row, k0 + g) : 0u;
        const bool h = (e & F_BH) && S.p_type[e & NB_IDX] == 1000;
        hit = ((__ballot(h) >> gbit) & ((1u << GROUP) - 1u)) != 0;   // the group agrees
    }
    if (g == 0) out[i] = hit ? 1 : 0;
}
int ibm_near_build(sph_ctx* c) {
    if (c->ibm_near_gen == c->generation && c->ibm_near) return 0;
    if (!c->ibm_near) SPH_TRY(dalloc(c, &c->ibm_near, (size_t)c->cap));
    if (c->n > 0) {
        hipLaunchKernelGGL(k_ibm_near, dim3(grid1((long long)c->n * GROUP)), dim3(BLOCK), 0, c->stream, c->n, c->sview(), c->nlist(),
                           c->ibm_near);
        SPH_TRY(launch_check(c, "ibm_near"));
    }
    c->ibm_near_gen = c->generation;
    return 0;
}

// The distinct particles of the Neumann pairs (a thin layer of fluid along
// walls, lid and buildings) and the pairs as indices into that set.
__global__ void __launch_bounds__(BLOCK) k_zero_i32(int n, int* a) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = 0;
}
__global__ void __launch_bounds__(BLOCK) k_nms_mark(long long m, const int* ent, int* mark) {
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < m) mark[ent[e]] = 1;
}
__global__ void __launch_bounds__(BLOCK) k_nms_list(int n, const int* mark, const int* idx, int* set) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && mark[i]) set[idx[i]] = i;
}
__global__ void __launch_bounds__(BLOCK) k_nms_remap(long long m, const int* ent, const int* idx, int* cent) {
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e < m) cent[e] = idx[ent[e]];
}
static int neumann_set(sph_ctx* c, long long total) {
    const int n = c->n;
    int *mark = nullptr, *idx = nullptr;
    SPH_TRY(dalloc(c, &mark, n));
    SPH_TRY(dalloc(c, &idx, n));
    hipLaunchKernelGGL(k_zero_i32, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, mark);
    hipLaunchKernelGGL(k_nms_mark, dim3(grid1(total)), dim3(BLOCK), 0, c->stream, total, (const int*)c->nmp_ent, mark);
    SPH_TRY(launch_check(c, "neumann_set_mark"));
    int nset = 0;
    SPH_TRY(exclusive_scan_i32(c, mark, idx, n, &nset));
    SPH_TRY(dalloc(c, &c->nm_set, (size_t)std::max(1, nset)));
    SPH_TRY(dalloc(c, &c->nmp_cent, (size_t)total));
    SPH_TRY(dalloc(c, &c->nm_rec, (size_t)std::max(1, nset) * NMREC_FLOATS));
    hipLaunchKernelGGL(k_nms_list, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, (const int*)mark, (const int*)idx,
                       c->nm_set);
    hipLaunchKernelGGL(k_nms_remap, dim3(grid1(total)), dim3(BLOCK), 0, c->stream, total, (const int*)c->nmp_ent,
                       (const int*)idx, c->nmp_cent);
    SPH_TRY(launch_check(c, "neumann_set"));
    dfree(c, mark);
    dfree(c, idx);
    c->nm_nset = nset;
    return 0;
}

int neumann_pairs(sph_ctx* c) {
    dfree(c, c->nmp_off);
    dfree(c, c->nmp_ent);
    dfree(c, c->nmp_cent);
    dfree(c, c->nm_set);
    dfree(c, c->nm_rec);
    c->nmp_off = nullptr;
    c->nmp_ent = nullptr;
    c->nmp_cent = nullptr;
    c->nm_set = nullptr;
    c->nm_rec = nullptr;
    c->nm_nset = 0;
    const int m = c->nm_count;
    if (m > 0 && c->nm_list) {
        const bool mixed = c->prm.precision == SPH_MIXED;
        const KConst kc{c->prm.kernel_type, c->prm.kappa, c->c_pi15};
        int* cnt = nullptr;
        long long* wide = nullptr;
        long long total = 0;
        SPH_TRY(dalloc(c, &cnt, m));
        SPH_TRY(dalloc(c, &wide, m));
        SPH_TRY(dalloc(c, &c->nmp_off, (size_t)m + 1));
        if (mixed)
            hipLaunchKernelGGL((k_nmp_build<float, false>), dim3(m), dim3(64), 0, c->stream, c->pview(), c->grid(), kc,
                               c->prm.L2, (const int*)c->nm_list, m, cnt, (const long long*)nullptr, (int*)nullptr);
        else
            hipLaunchKernelGGL((k_nmp_build<double, false>), dim3(m), dim3(64), 0, c->stream, c->pview(), c->grid(),
                               kc, c->prm.L2, (const int*)c->nm_list, m, cnt, (const long long*)nullptr, (int*)nullptr);
        SPH_TRY(launch_check(c, "neumann_pairs_count"));
        hipLaunchKernelGGL(k_nmp_widen, dim3(grid1(m)), dim3(BLOCK), 0, c->stream, m, (const int*)cnt, wide);
        SPH_TRY(launch_check(c, "neumann_pairs_widen"));
        SPH_TRY(exclusive_scan_i64(c, wide, c->nmp_off, m, &total));
        SPH_HIP(c, hipMemcpyAsync(c->nmp_off + m, &total, sizeof(long long), hipMemcpyHostToDevice, c->stream));
        SPH_TRY(dalloc(c, &c->nmp_ent, (size_t)std::max(1LL, total)));
        if (mixed)
            hipLaunchKernelGGL((k_nmp_build<float, true>), dim3(m), dim3(64), 0, c->stream, c->pview(), c->grid(), kc,
                               c->prm.L2, (const int*)c->nm_list, m, (int*)nullptr, (const long long*)c->nmp_off,
                               c->nmp_ent);
        else
            hipLaunchKernelGGL((k_nmp_build<double, true>), dim3(m), dim3(64), 0, c->stream, c->pview(), c->grid(),
                               kc, c->prm.L2, (const int*)c->nm_list, m, (int*)nullptr, (const long long*)c->nmp_off,
                               c->nmp_ent);
        SPH_TRY(launch_check(c, "neumann_pairs_fill"));
        SPH_HIP(c, hipStreamSynchronize(c->stream));   // total lives on this frame
        dfree(c, cnt);
        dfree(c, wide);
        if (mixed && c->pos_f32 && !c->prm.ale_positions && total > 0) SPH_TRY(neumann_set(c, total));
    }
    c->nmp_gen = c->generation;
    c->nmp_for = c->nm_list;
    c->nmp_prec = c->prm.precision;
    return 0;
}

static int run_neumann(Eng& e, int which, int only_count0) {
    SEGL("snapshot", k_snapshot, which, 1);
    if (mixed_of(e)) {
        tune_fixed(e, TK_NEUMANN, WAVE_BLOCK);
        BOUNDW("neumann", NM_LANES, k_neumann_mixed, which, only_count0);
        return 0;
    }
    tune_fixed(e, TK_NEUMANN, NM_BLOCK);
    Shape sh;   // a block per boundary particle of each case
    SPH_TRY(shape(e, 3, NM_BLOCK, &sh));
    if (sh.grid > 0) {
        SPH_TRY(prof_begin(e, "neumann", 0.0));
        hipLaunchKernelGGL(k_neumann, dim3(sh.grid), dim3(NM_BLOCK), 0, e.st, Seg{e.d_desc, sh.tab}, which, only_count0);
        SPH_TRY(launch_check(&e, "neumann"));
        SPH_TRY(prof_end(e));
    }
    return 0;
}
static int run_outlet(Eng& e, int which) {
    SEGL("snapshot", k_snapshot, which, 0);
    SEGL("outlet", k_outlet, which);
    return 0;
}
static int run_periodic(Eng& e, int which) {
    SEGL("snapshot", k_snapshot, which, 0);
    SEGL("periodic", k_periodic, which);
    return 0;
}
static int run_freeslip(Eng& e, int which) {
    if (mixed_of(e)) BOUNDL("freeslip", k_freeslip_mixed, which);   // the lid's particles among the boundary ones
    else BOUNDL("freeslip", k_freeslip, which);
    return 0;
}

// Neighbour records of every case of the step, from its working state as
// it is now; run before each pass that gathers from them.
int pack_records(Eng& e, int which) {
    if (which == REC_PRE) {
        bool any = false;
        for (size_t k = 0; k < e.cs.size(); k++) any |= e.h_desc[k].crec_adv != nullptr;
        if (any) SEGL("pack_records", k_pack_records<REC_PRE>);
        return 0;
    }
    if (which == REC_PQ) SEGL("pack_records", k_pack_records<REC_PQ>);
    else if (which == REC_VEL_PQ) SEGL("pack_records", k_pack_records<REC_VEL_PQ>);
    else SEGL("pack_records", k_pack_records<REC_ALL>);
    return 0;
}

// KERNEL_clc_IB_normal_vector3D, functions_PREP.cuh:923-1015 (count == 0,
// ISPH_Calc.cuh:70-74): markers within ib_face_tol of a face plane get -1 / +1
// on that axis (the upper plane wins a tie, as it is tested last), normalised
// in float with IEEE round-to-nearest square root and division.  In
// SPH_IBN_REFERENCE mode a step with count > 0 writes zero normals, the
// values the reference's per-step part3 reset leaves (ISPH_Calc.cuh:61).
__global__ void __launch_bounds__(BLOCK) k_ib_normals(Seg sg) {
    SEG_PARTICLE(sg);
    const sph_params& pr = cd.pr;
    if (pr.ib_normals == SPH_IBN_UPLOADED) return;
    if (cd.count > 0 && pr.ib_normals == SPH_IBN_PLANES) return;
    const PView S = cd.S;
    if (S.p_type[i] < 1000) return;
    float nx = 0.0f, ny = 0.0f, nz = 0.0f;
    if (cd.count == 0) {
        const double xi = S.x[i], yi = S.y[i], zi = S.z[i], tol = pr.ib_face_tol;
        if (fabs(xi - pr.ib_face_xlo) < tol) nx = -1.0f;
        if (fabs(xi - pr.ib_face_xhi) < tol) nx = 1.0f;
        if (fabs(yi - pr.ib_face_ylo) < tol) ny = -1.0f;
        if (fabs(yi - pr.ib_face_yhi) < tol) ny = 1.0f;
        if (fabs(zi - pr.ib_face_zlo) < tol) nz = -1.0f;
        if (fabs(zi - pr.ib_face_zhi) < tol) nz = 1.0f;
    }
    const float mag = __fsqrt_rn(nx * nx + ny * ny + nz * nz);
    const QView Q = cd.Q;
    if ((double)mag > 1e-9) {
        Q.nx[i] = (double)__fdiv_rn(nx, mag);
        Q.ny[i] = (double)__fdiv_rn(ny, mag);
        Q.nz[i] = (double)__fdiv_rn(nz, mag);
    } else {
        Q.nx[i] = 0.0; Q.ny[i] = 0.0; Q.nz[i] = 0.0;
    }
}

// The host-side choices of step_physics_front, one bit each.
long long step_physics_front_key(const Eng& e) {
    long long key = mixed_of(e) ? 1 : 0;
    bool count0 = false, gc = false, nrm = false, scal = false, compact = false;
    for (size_t k = 0; k < e.cs.size(); k++) {
        const sph_ctx* c = e.cs[k];
        count0 |= e.h_desc[k].count == 0;
        gc |= !e.h_desc[k].gc_fresh;
        const int m = c->prm.ib_normals;
        nrm |= m == SPH_IBN_REFERENCE || (m == SPH_IBN_PLANES && e.h_desc[k].count == 0);
        scal |= c->prm.con_solve || c->prm.concn_solve || c->prm.boussinesq_solve;
        compact |= e.h_desc[k].crec_adv != nullptr;
    }
    return key | (count0 ? 2 : 0) | (gc ? 4 : 0) | (nrm ? 8 : 0) | (scal ? 16 : 0) | (compact ? 32 : 0) |
           (e.tile_lanes ? 64 : 0);
}
long long step_physics_back_key(const Eng& e) {
    bool ale = false;
    for (const sph_ctx* c : e.cs) ale |= c->prm.ale_positions != 0;
    return (mixed_of(e) ? 1 : 0) | (ale ? 2 : 0) | (e.tile_lanes ? 4 : 0);
}

// Everything of SOPHIA_single_ISPH before the pressure solve
// (ISPH_Calc.cuh:20-132).  The count==0 neighbour searches have already run.
int step_physics_front(Eng& e) {
    const bool mixed = mixed_of(e);
    bool any_count0 = false;
    for (size_t k = 0; k < e.cs.size(); k++) any_count0 |= e.h_desc[k].count == 0;
    SEGL("step_begin", k_step_begin);
    bool any_nrm = false;   // a case whose marker normals this step sets
    for (size_t k = 0; k < e.cs.size(); k++) {
        const int m = e.cs[k]->prm.ib_normals;
        any_nrm |= m == SPH_IBN_REFERENCE || (m == SPH_IBN_PLANES && e.h_desc[k].count == 0);
    }
    if (any_nrm) SEGL("ib_normals", k_ib_normals);
    bool any_gc = false;
    for (size_t k = 0; k < e.cs.size(); k++) any_gc |= !e.h_desc[k].gc_fresh;
    if (any_gc) {
        if (mixed) SEGG("grad_corr", TK_GRAD_CORR, k_grad_corr_mixed);
        else SEGO("grad_corr", TK_GRAD_CORR, ord_doubles(GC_SUMS), k_grad_corr);
    }
    SPH_TRY(pack_records(e, REC_PRE));   // compact records for the strain pass
    if (mixed && e.tile_lanes) TILEL("prep", k_prep_tile, CREC_ADV_FLOATS);
    else if (mixed) {
        SEGG("prep", TK_PREP, k_prep_mixed);
        HEAVYL("prep_heavy", k_prep_heavy);
    } else SEGO("prep", TK_PREP, ord_doubles(PREP_SUMS), k_prep);
    if (mixed) BOUNDL("boundary3d", k_boundary3d_mixed);
    else BOUNDL("boundary3d", k_boundary3d);
    SEGL("most_self", k_most_self);
    SEGL("most_deposit", k_most_deposit);
    if (any_count0) SPH_TRY(run_neumann(e, 0, 1));
    SPH_TRY(pack_records(e, REC_ALL));
    bool scal = false;   // scalar transport or buoyancy in some case of the step
    for (sph_ctx* c : e.cs) scal |= c->prm.con_solve || c->prm.concn_solve || c->prm.boussinesq_solve;
    if (mixed) {
        if (e.tile_lanes) {
            if (scal) TILEL("advection", k_advection_tile<true>, CREC_ADV_FLOATS);
            else TILEL("advection", k_advection_tile<false>, CREC_ADV_FLOATS);
        } else if (scal) {
            SEGG("advection", TK_ADVECTION, k_advection_mixed<true>);
            HEAVYL("advection_heavy", k_advection_heavy<true>);
        } else {
            SEGG("advection", TK_ADVECTION, k_advection_mixed<false>);
            HEAVYL("advection_heavy", k_advection_heavy<false>);
        }
    } else {
        if (scal) SEGO("advection", TK_ADVECTION, ord_doubles(adv_sums<true>(), ADV_SECOND), k_advection<true>);
        else SEGO("advection", TK_ADVECTION, ord_doubles(adv_sums<false>(), ADV_SECOND), k_advection<false>);
    }
    SEGL("projection", k_projection);
    SPH_TRY(run_periodic(e, 0));
    SPH_TRY(run_freeslip(e, 0));
    return 0;
}

// Everything after the pressure solve (ISPH_Calc.cuh:143-214).
int step_physics_back(Eng& e) {
    const bool mixed = mixed_of(e);
    SPH_TRY(run_neumann(e, 0, 0));
    SPH_TRY(run_outlet(e, 0));
    SPH_TRY(pack_records(e, REC_PQ));   // pressures after the solve and the boundary passes
    if (mixed && e.tile_lanes) TILEL("pressure_force", k_pressure_force_tile, CREC_FLOATS);
    else if (mixed) {
        SEGG("pressure_force", TK_PRESSURE, k_pressure_force_mixed);
        HEAVYL("pressure_force_heavy", k_pressure_force_heavy);
    }
    else SEGO("pressure_force", TK_PRESSURE, ord_doubles(PF_SUMS), k_pressure_force);
    if (mixed) BOUNDL("ibm_force", k_ibm_force_mixed);
    else BOUNDL("ibm_force", k_ibm_force);
    if (mixed) SEGG("ibm_spread", TK_IBM_SPREAD, k_ibm_spread_mixed);
    else SEGO("ibm_spread", TK_IBM_SPREAD, ord_doubles(4), k_ibm_spread);
    SEGL("time_update", k_time_update);
    SPH_TRY(run_neumann(e, 1, 0));
    SPH_TRY(run_outlet(e, 1));
    SPH_TRY(run_periodic(e, 1));
    SPH_TRY(run_freeslip(e, 1));
    bool ale = false;
    for (sph_ctx* c : e.cs) ale |= c->prm.ale_positions != 0;
    if (ale) SEGL("commit_positions", k_commit_positions);
    return 0;
}

int stats_run(sph_ctx* c, float* umax, float* drho, float* fmax_) {
    const int n = c->n;
    unsigned* acc = (unsigned*)c->stat_buf;
    SPH_HIP(c, hipMemsetAsync(acc, 0, 3 * sizeof(unsigned), c->stream));
    hipLaunchKernelGGL(k_stats, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, c->pview(), c->s2view(), c->qview(), acc);
    SPH_TRY(launch_check(c, "stats"));
    hipLaunchKernelGGL(k_stats_final, dim3(1), dim3(64), 0, c->stream, (const unsigned*)acc, c->stat_buf + 4);
    SPH_TRY(launch_check(c, "stats_final"));
    float h[3];
    SPH_HIP(c, hipMemcpyAsync(h, c->stat_buf + 4, 3 * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    SPH_HIP(c, hipStreamSynchronize(c->stream));
    *umax = h[0]; *drho = h[1]; *fmax_ = h[2];
    return 0;
}

// ---- statistics without allocation (sph_stats_noalloc) -------------------
// Per-workgroup maxima go behind the context's accumulators (stat_buf, sized for
// them when the context is made) and a one-workgroup fold reduces them, so the
// call needs no device allocation, no memset and no atomics, and contexts share
// nothing.

// The maxima of k_stats for this workgroup's particles, stored at part[3b..3b+2].
__global__ void __launch_bounds__(BLOCK) k_stats_part(int n, PView P, P2View S2, QView Q, unsigned* part) {
    __shared__ unsigned s[3][BLOCK];
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    float a = 0, b = 0, c = 0;
    if (i < n && !(P.p_type[i] == 0 || P.i_type[i] >= 2)) {
        a = (float)sqrt(P.ux[i] * P.ux[i] + P.uy[i] * P.uy[i] + P.uz[i] * P.uz[i]);
        b = (float)((P.rho[i] - S2.rho_ref[i]) / S2.rho_ref[i] * 100.0);
        c = (float)Q.ftotal[i];
    }
    s[0][threadIdx.x] = i < n ? f2ord(a) : 0u;
    s[1][threadIdx.x] = i < n ? f2ord(b) : 0u;
    s[2][threadIdx.x] = i < n ? f2ord(c) : 0u;
    __syncthreads();
    for (int off = BLOCK / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off)
            for (int q = 0; q < 3; q++) s[q][threadIdx.x] = max(s[q][threadIdx.x], s[q][threadIdx.x + off]);
        __syncthreads();
    }
    if (threadIdx.x < 3) part[3 * blockIdx.x + threadIdx.x] = s[threadIdx.x][0];
}
// One workgroup: the maxima over the nb partials (starting from 0, as the
// zeroed accumulator of k_stats does), as floats into out[0..2].
__global__ void __launch_bounds__(BLOCK) k_stats_fold(int nb, const unsigned* part, float* out) {
    __shared__ unsigned s[3][BLOCK];
    unsigned a = 0u, b = 0u, c = 0u;
    for (int k = threadIdx.x; k < nb; k += BLOCK) {
        a = max(a, part[3 * k]);
        b = max(b, part[3 * k + 1]);
        c = max(c, part[3 * k + 2]);
    }
    s[0][threadIdx.x] = a; s[1][threadIdx.x] = b; s[2][threadIdx.x] = c;
    __syncthreads();
    for (int off = BLOCK / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off)
            for (int q = 0; q < 3; q++) s[q][threadIdx.x] = max(s[q][threadIdx.x], s[q][threadIdx.x + off]);
        __syncthreads();
    }
    if (threadIdx.x < 3) out[threadIdx.x] = ord2f(s[threadIdx.x][0]);
}

int stats_run_noalloc(sph_ctx* c, float* umax, float* drho, float* fmax_) {
    const int n = c->n;
    if ((long long)n > NA_STATS_MAX_N)
        return fail(c, SPH_E_ARG, "sph_stats_noalloc: " + std::to_string(n) + " particles exceed its bound of " +
                                      std::to_string(NA_STATS_MAX_N) + " (use sph_stats)");
    unsigned* const part = (unsigned*)c->stat_buf + STAT_PARTS;
    const unsigned nb = grid1(n);
    hipLaunchKernelGGL(k_stats_part, dim3(nb), dim3(BLOCK), 0, c->stream, n, c->pview(), c->s2view(), c->qview(), part);
    SPH_TRY(launch_check(c, "stats_part"));
    float* res = c->stat_buf + 4;
    hipLaunchKernelGGL(k_stats_fold, dim3(1), dim3(BLOCK), 0, c->stream, (int)nb, (const unsigned*)part, res);
    SPH_TRY(launch_check(c, "stats_fold"));
    float h[3];
    SPH_HIP(c, hipMemcpyAsync(h, res, 3 * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    SPH_HIP(c, hipStreamSynchronize(c->stream));
    *umax = h[0]; *drho = h[1]; *fmax_ = h[2];
    return 0;
}

}  // namespace sph
