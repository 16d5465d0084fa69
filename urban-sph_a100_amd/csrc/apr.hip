// Adaptive particle refinement (APR): cell-based 1 -> 8 splitting.
//
//   KERNEL_APR_condition3D_cell, splitting branch  functions_APR.cuh:270-330  -> k_apr_pick
//   Cell_index (prefix sum of the cell flags)     functions_APR_etc.cuh:366   -> k_apr_pick, k_apr_list
//   KERNEL_cell_APR_3D, splitting branch          functions_APR.cuh:420-500  -> k_apr_split
//   Particle_refinement_cell                      functions_APR_etc.cuh:354-375 -> sph_apr_refine
//
// A particle's refinement level is log8(m_ref / m).  In every occupied cell
// the first particle (in cell order) whose target level exceeds its level
// by at least 0.75 is split into 8 children at +-a along each axis,
// a = cbrt(m / rho) / 4, rounded to float positions as the reference's
// float records hold them, with m/8, vol/8 and h/2 (when apr_h_change),
// every other field copied.  Children of the k-th splitting cell (ascending cell
// index) go to n + 8k..n + 8k + 7 in the reference's order; the parent
// becomes a dummy (i_type 3).  One split per cell per pass; the neighbour
// search runs again after each pass.
//
// The reference keeps the target level (M_num) and the split flag
// (apr_cond) in its particle record, but both are commented out of the
// compiled record (class_Cuda_Particle_Array.cuh:37-43); here the target
// level is a per-particle array of the context, inherited by the children.
#include <climits>

#include "flags.h"
#include "sph_internal.h"
#include "sph_math.h"

namespace sph {

// Cube root by Newton's method on the mantissa.  The same IEEE operations
// run on every device, so children's positions agree bit for bit with any
// other evaluation of this routine.
__device__ __forceinline__ double apr_cbrt(double v) {
    int e = 0;
    double m = frexp(v, &e);          // v = m 2^e, m in [0.5, 1)
    const int r = ((e % 3) + 3) % 3;
    m = ldexp(m, r);                  // m in [0.5, 4), e - r divisible by 3
    e -= r;
    double y = 1.0;
#pragma unroll
    for (int it = 0; it < 8; it++) y = y - (y * y * y - m) / (3.0 * y * y);
    return ldexp(y, e / 3);
}

// The first particle of each cell (in cell order) that wants to split: a
// thread per particle, the lowest index of a cell kept (a refined cell holds
// hundreds of particles, which a thread per cell walked one by one: 205 us a pass of
// the 226 k refined canyon).
__global__ void __launch_bounds__(BLOCK) k_apr_first(int ncells, int* pick) {
    const int cell = blockIdx.x * blockDim.x + threadIdx.x;
    if (cell < ncells) pick[cell] = INT_MAX;
}
__global__ void __launch_bounds__(BLOCK) k_apr_want(int n, int ncells, const int* keys, PView P, const double* target,
                                                    int* pick) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const int cell = keys[j];
    if (cell < 0 || cell >= ncells) return;   // a dummy
    const double level = log(P.m_ref[j] / P.m[j]) / log(8.0);
    if (target[j] - level >= 0.75) atomicMin(&pick[cell], j);
}
// the split loop passes over a non-fluid particle whose target exceeds 2, and
// the condition marked only the cell's first one (functions_APR.cuh:423).
// rank: a splitting cell's number within its tile of RS_TILE cells, -1 elsewhere;
// sums: the tiles' splitting cells.
__global__ void __launch_bounds__(BLOCK) k_apr_pick(int ncells, PView P, const double* target, const int* pick,
                                                    int* rank, int* sums) {
    __shared__ int wsum[BLOCK / 64];
    const int t = threadIdx.x, lane = t & 63, base = blockIdx.x * RS_TILE + t * RS_ITEMS;
    int flag[RS_ITEMS], s = 0;
#pragma unroll
    for (int k = 0; k < RS_ITEMS; k++) {
        const int j = base + k < ncells ? pick[base + k] : INT_MAX;
        flag[k] = j != INT_MAX && !(P.p_type[j] != 1 && target[j] > 2.0) ? 1 : 0;
        s += flag[k];
    }
    int up = s;   // inclusive over the wave
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int a = __shfl_up(up, off);
        if (lane >= off) up += a;
    }
    if (lane == 63) wsum[t >> 6] = up;
    __syncthreads();
    int run = up - s;
    for (int w = 0; w < (t >> 6); w++) run += wsum[w];
    if (t == BLOCK - 1) sums[blockIdx.x] = run + s;
#pragma unroll
    for (int k = 0; k < RS_ITEMS; k++) {
        if (base + k < ncells) rank[base + k] = flag[k] ? run : -1;
        run += flag[k];
    }
}
// The splitting particles in ascending cell order, and their number; the picks
// are cleared for the next pass.  A block's cells lie in one tile: it adds the sums
// of the tiles before.  (Flags, a scan of three launches and this list were five
// launches a pass, two of them after the host had waited for the number; a pass is
// bound by the host's 6-15 us a launch: a pass of a refined 150 k cloud is 410 -> 280 us of
// trace with the sort's and the cells' fewer launches, its refinement and two
// steps 61.3 -> 59.6 ms)
__global__ void __launch_bounds__(BLOCK) k_apr_list(int ncells, int ntiles, const int* rank, const int* sums, int* pick,
                                                    int* list, int* nsplit) {
    __shared__ int part[BLOCK / 64];
    const int t = threadIdx.x, cell = blockIdx.x * BLOCK + t, tile = blockIdx.x * BLOCK / RS_TILE;
    auto sum_to = [&](int end) {   // of sums[0 .. end), in every thread
        int s = 0;
        for (int q = t; q < end; q += BLOCK) s += sums[q];
#pragma unroll
        for (int off = 32; off; off >>= 1) s += __shfl_xor(s, off);
        __syncthreads();
        if ((t & 63) == 0) part[t >> 6] = s;
        __syncthreads();
        s = 0;
        for (int w = 0; w < BLOCK / 64; w++) s += part[w];
        return s;
    };
    if (blockIdx.x == 0) {
        const int all = sum_to(ntiles);
        if (t == 0) *nsplit = all;
    }
    const int before = sum_to(tile);
    if (cell >= ncells) return;
    const int r = rank[cell];
    if (r >= 0) list[before + r] = pick[cell];
    pick[cell] = INT_MAX;
}

constexpr int APR_MAX_F64 = 64;
struct AprFields {
    double* f[APR_MAX_F64];
    int* iv[SPH_I_COUNT];
    int nf;
    double *x, *y, *z, *m, *vol, *h, *rho;
};

// A thread per child (the children of consecutive splits are consecutive, so
// every field is written in whole lines).  The parent becomes a dummy once its
// children hold its fields: they are eight consecutive lanes of one wave, whose
// loads all precede the store.  SPLIT_U fields' loads are in flight: one field
// after another took 21 us a pass, now 10 (59.6 -> 59.0 ms).
constexpr int SPLIT_U = 16;
__global__ void __launch_bounds__(BLOCK) k_apr_split(int nsplit, const int* list, int n0, AprFields F, int h_change) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x, k = t & 7;
    if (t >= 8 * nsplit) return;
    const int j = list[t >> 3], c = n0 + t;
    const double xm = F.x[j], ym = F.y[j], zm = F.z[j];
    const double a = 0.25 * apr_cbrt(F.m[j] / F.rho[j]);
    for (int f0 = 0; f0 < F.nf; f0 += SPLIT_U) {
        double v[SPLIT_U];
#pragma unroll
        for (int u = 0; u < SPLIT_U; u++)
            if (f0 + u < F.nf) v[u] = F.f[f0 + u][j];
#pragma unroll
        for (int u = 0; u < SPLIT_U; u++)
            if (f0 + u < F.nf) F.f[f0 + u][c] = v[u];
    }
    int w[SPH_I_COUNT];
#pragma unroll
    for (int f = 0; f < SPH_I_COUNT; f++) w[f] = F.iv[f][j];
#pragma unroll
    for (int f = 0; f < SPH_I_COUNT; f++) F.iv[f][c] = w[f];
    // child order of functions_APR.cuh:440-478: x +,+,+,+,-,-,-,-;
    // y +,+,-,-,+,+,-,-; z +,-,+,-,+,-,+,-.  The reference stores the
    // children's positions in its float records (functions_APR.cuh:
    // 544-590): rounded to float here too, so a refined case's positions
    // stay float values
    F.x[c] = (double)(float)(k < 4 ? xm + a : xm - a);
    F.y[c] = (double)(float)((k & 2) ? ym - a : ym + a);
    F.z[c] = (double)(float)((k & 1) ? zm - a : zm + a);
    F.m[c] = 0.125 * F.m[j];
    F.vol[c] = 0.125 * F.vol[j];
    if (h_change) F.h[c] = 0.5 * F.h[j];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (k == 0) F.iv[SPH_I_I_TYPE][j] = 3;
}

int apr_refine(sph_ctx* c, const double* target, int max_passes, int* n_out) {
    const int ncells = c->dom.num_cells - 1;
    if (!c->apr_target) {
        SPH_TRY(dalloc(c, &c->apr_target, c->cap));
        SPH_HIP(c, hipMemsetAsync(c->apr_target, 0, sizeof(double) * (size_t)c->cap, c->stream));
    }
    if (target)
        SPH_HIP(c, hipMemcpyAsync(c->apr_target, target, sizeof(double) * (size_t)c->n, hipMemcpyHostToDevice, c->stream));
    int *rank = nullptr, *pick = nullptr, *list = nullptr, *sums = nullptr;
    const int ntiles = (ncells + RS_TILE - 1) / RS_TILE;
    SPH_TRY(dalloc(c, &list, ncells));
    SPH_TRY(dalloc(c, &rank, ncells));
    SPH_TRY(dalloc(c, &pick, ncells));
    SPH_TRY(dalloc(c, &sums, ntiles));
    SPH_TRY(back_slot(c));
    hipLaunchKernelGGL(k_apr_first, dim3(grid1(ncells)), dim3(BLOCK), 0, c->stream, ncells, pick);
    int rc = launch_check(c, "apr_first");
    bool split_any = false;
    for (int pass = 0; pass < max_passes && rc == 0; pass++) {
        hipLaunchKernelGGL(k_apr_want, dim3(grid1(c->n)), dim3(BLOCK), 0, c->stream, c->n, ncells, (const int*)c->keys,
                           c->pview(), (const double*)c->apr_target, pick);
        hipLaunchKernelGGL(k_apr_pick, dim3(ntiles), dim3(BLOCK), 0, c->stream, ncells, c->pview(),
                           (const double*)c->apr_target, (const int*)pick, rank, sums);
        hipLaunchKernelGGL(k_apr_list, dim3(grid1(ncells)), dim3(BLOCK), 0, c->stream, ncells, ntiles, (const int*)rank,
                           (const int*)sums, pick, list, (int*)c->back);
        if ((rc = launch_check(c, "apr_pick"))) break;
        int nsplit = 0;
        const hipError_t he = hipStreamSynchronize(c->stream);
        if (he != hipSuccess) { rc = fail(c, SPH_E_HIP, hipGetErrorString(he)); break; }
        nsplit = *(const int*)c->back;
        if (nsplit == 0) break;
        if ((long long)c->n + 8LL * nsplit > c->cap) {
            rc = fail(c, SPH_E_NOMEM, "APR needs room for " + std::to_string(c->n + 8LL * nsplit) +
                                          " particles; create the context with a larger n_part2");
            break;
        }
        AprFields F{};
        for (int f = 0; f < SPH_F_COUNT_F64 + 3; f++)
            if (c->pf[f]) F.f[F.nf++] = c->pf[f];
        for (int f = 0; f < 10; f++) F.f[F.nf++] = c->p2[f];
        for (int f = 15; f < 18; f++) F.f[F.nf++] = c->q[f];
        F.f[F.nf++] = c->apr_target;
        for (int f = 0; f < SPH_I_COUNT; f++) F.iv[f] = c->pi[f];
        F.x = c->pf[SPH_F_X]; F.y = c->pf[SPH_F_Y]; F.z = c->pf[SPH_F_Z]; F.m = c->pf[SPH_F_M];
        F.vol = c->pf[SPH_F_VOL]; F.h = c->pf[SPH_F_H]; F.rho = c->pf[SPH_F_RHO];
        hipLaunchKernelGGL(k_apr_split, dim3(grid1(8LL * nsplit)), dim3(BLOCK), 0, c->stream, nsplit, (const int*)list,
                           c->n, F, c->prm.apr_h_change);
        if ((rc = launch_check(c, "apr_split"))) break;
        c->n += 8 * nsplit;   // the children's positions are float values like their parents'
        dfree(c, c->porder);   // the pass order covers the old count; the next list rebuilds it
        c->porder = nullptr;
        ppe_free(c);
        if ((rc = set_ncell_run(c))) break;
        // the next pass needs only the cells; the neighbour list is built
        // once after the last pass, on the cells and order of its search
        rc = nnps_run(c, false);
        split_any = true;
    }
    if (split_any) {   // also after a failed pass: the lists match the particles there are
        const int lrc = nnps_list(c);
        if (rc == 0) rc = lrc;
    }
    dfree(c, sums);
    dfree(c, rank);
    dfree(c, pick);
    dfree(c, list);
    if (n_out) *n_out = c->n;
    return rc;
}

}  // namespace sph
