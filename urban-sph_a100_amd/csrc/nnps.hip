// Neighbour search of the count==0 step on MI355X (ISPH_Calc.cuh:23-52):
//   KERNEL_index_particle_to_cell  functions_NNPS.cuh:879-907  -> k_hash
//   cub::DeviceRadixSort::SortPairs ISPH_Calc.cuh:33           -> radix_sort
//   KERNEL_reorder (start/end)     functions_NNPS.cuh:813-838  -> k_cells
//   KERNEL_reorder (gather)        functions_NNPS.cuh:840-843  -> permute
// plus the per-particle neighbour list that the per-step passes walk
// (the reference rescans the cell window in every pass).
//
// The sort is a stable least-significant-digit radix sort over only the
// ceil(log2(num_cells+1)) key bits, 8 bits per pass.  Each 256-thread tile
// of 2048 keys ranks its keys with wave64 ballots (a match-any over the
// digit bits) and LDS per-wave digit counters, so equal digits keep input
// order and the result equals a stable sort.
#include "flags.h"
#include <algorithm>
#include <climits>
#include <cstring>
#include <utility>

#include "sph_internal.h"
#include "sph_math.h"

namespace sph {

// ------------------------------------------------------------------------
// KERNEL_set_ncell, functions_NNPS.cuh:943-955
__global__ void __launch_bounds__(BLOCK) k_set_ncell(int n, const int* i_type, const double* h, const double* h_ref,
                                                     int* ncell) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (i_type[i] == 3) return;
    ncell[i] = (int)(1.0 * ceilf(2.0f / (float)(h_ref[i] / h[i])));
}

// KERNEL_index_particle_to_cell, functions_NNPS.cuh:879-907 (float binning)
__global__ void __launch_bounds__(BLOCK) k_hash(int n, sph_domain d, const int* i_type, const double* x,
                                                const double* y, const double* z, int* keys, int* vals) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int key;
    if (i_type[i] == 3) key = d.num_cells;
    else {
        Cell c = bin_cell(d, x[i], y[i], z[i]);
        key = c.i + d.NI * c.j + d.NI * d.NJ * c.k;
    }
    keys[i] = key;
    vals[i] = i;
}

// ------------------------------------------------------------------------
// radix sort

__global__ void __launch_bounds__(BLOCK) k_rs_hist(const int* keys, int n, int shift, int ntiles, int* hist) {
    __shared__ int h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    long long base = (long long)blockIdx.x * RS_TILE;
#pragma unroll
    for (int k = 0; k < RS_ITEMS; k++) {
        long long idx = base + k * BLOCK + threadIdx.x;
        if (idx < n) atomicAdd(&h[(keys[idx] >> shift) & 255], 1);
    }
    __syncthreads();
    hist[threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// offs: the histogram's prefixes within its scan tiles, sums: the tiles' sums
// (nsums of them).  Each block adds the sums of the tiles before its entries:
// thread t scans the t-th of 256 runs of sums, and a digit's base is the runs
// before its tile's and the rest of that run.  As launches of their own the scan
// of the sums and the addition were two of five a digit, of 2-3 us each with the
// host's 6-15 us between them where a refinement pass searches 150 k particles.
__global__ void __launch_bounds__(BLOCK) k_rs_scatter(const int* kin, const int* vin, int* kout, int* vout, int n,
                                                      int shift, int ntiles, const int* offs, const int* sums,
                                                      int nsums) {
    __shared__ int cnt[256];
    __shared__ int wc[BLOCK / 64][256];
    __shared__ int boff[256];
    __shared__ int run[BLOCK];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    cnt[tid] = 0;
    const int entry = tid * ntiles + blockIdx.x, tile = entry / RS_TILE, per = (nsums + BLOCK - 1) / BLOCK;
    int base_d = offs[entry];
    int s = 0;
    for (int q = tid * per; q < min(nsums, (tid + 1) * per); q++) s += sums[q];
    run[tid] = s;
    __syncthreads();
    for (int off = 1; off < BLOCK; off <<= 1) {
        const int a = tid >= off ? run[tid - off] : 0;
        __syncthreads();
        run[tid] += a;
        __syncthreads();
    }
    if (tile >= per) base_d += run[tile / per - 1];
    for (int q = tile / per * per; q < tile; q++) base_d += sums[q];
    boff[tid] = base_d;
#pragma unroll
    for (int q = 0; q < BLOCK / 64; q++) wc[q][tid] = 0;
    __syncthreads();
    long long base = (long long)blockIdx.x * RS_TILE;
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int k = 0; k < RS_ITEMS; k++) {
        long long idx = base + k * BLOCK + tid;
        bool valid = idx < n;
        int key = valid ? kin[idx] : 0;
        int val = valid ? vin[idx] : 0;
        int dg = valid ? ((key >> shift) & 255) : 256;
        unsigned long long peers = ~0ull;
#pragma unroll
        for (int b = 0; b < 9; b++) {
            int bit = (dg >> b) & 1;
            unsigned long long bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        int wrank = __popcll(peers & lt);
        int wcount = __popcll(peers);
        int leader = __ffsll((long long)peers) - 1;
        if (valid && lane == leader) wc[w][dg] = wcount;
        __syncthreads();
        if (valid) {
            int pre = cnt[dg];
            for (int q = 0; q < w; q++) pre += wc[q][dg];
            int pos = boff[dg] + pre + wrank;
            kout[pos] = key;
            vout[pos] = val;
        }
        __syncthreads();
        int add = 0;
#pragma unroll
        for (int q = 0; q < BLOCK / 64; q++) { add += wc[q][tid]; wc[q][tid] = 0; }
        cnt[tid] += add;
        __syncthreads();
    }
}

// Up to SMALL_N pairs in one launch, in place: one workgroup, each wave a run of
// the pairs in order, a digit at a time.  A wave ranks its pairs by ballots and
// counts its digits in its own row of wc; the rows become bases (digit by digit,
// wave by wave); keys and original places move through LDS and the values follow
// at the end.  Three launches a digit of 5-9 us each, with the host's launches
// between them, were most of a small sort (the block tables of every search and
// the coarse multigrid levels sort some thousand pairs): the 4 k FP64 box 1.98 ->
// 1.86 ms, the 55 k boxes 5.03 -> 4.93 and 8.85 -> 8.57 ms, the moving 300 k case
// 39.6 -> 39.2 ms.
constexpr int SMALL_T = 1024, SMALL_W = SMALL_T / 64, SMALL_ITEMS = 8, SMALL_N = SMALL_T * SMALL_ITEMS;
__global__ void __launch_bounds__(SMALL_T) k_sort_small(int* keys, int* vals, int n, int digits) {
    __shared__ int lk[SMALL_N];
    __shared__ unsigned short li[SMALL_N], wc[SMALL_W][256];
    __shared__ int wsum[4], base[256];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int per = ((n + SMALL_T - 1) / SMALL_T) * 64;   // a wave's run
    const unsigned long long lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int key[SMALL_ITEMS], at[SMALL_ITEMS], rank[SMALL_ITEMS];
#pragma unroll
    for (int r = 0; r < SMALL_ITEMS; r++) {
        const int i = w * per + r * 64 + lane;
        at[r] = i;
        key[r] = r * 64 < per && i < n ? keys[i] : 0;
    }
    for (int p = 0; p < digits; p++) {
        for (int q = t; q < SMALL_W * 256; q += SMALL_T) (&wc[0][0])[q] = 0;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < SMALL_ITEMS; r++) {
            if (r * 64 >= per) break;
            const bool valid = w * per + r * 64 + lane < n;
            const int dg = (key[r] >> (8 * p)) & 255;
            unsigned long long peers = __ballot(valid);
            if (!valid) peers = ~peers;
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const int bit = (dg >> b) & 1;
                const unsigned long long bal = __ballot(bit);
                peers &= bit ? bal : ~bal;
            }
            const int before = wc[w][dg];
            rank[r] = before + __popcll(peers & lt);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            if (valid && lane == __ffsll((long long)peers) - 1) wc[w][dg] = (unsigned short)(before + __popcll(peers));
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        int sum = 0, up = 0;
        if (t < 256) {
            for (int q = 0; q < SMALL_W; q++) {
                const int v = wc[q][t];
                wc[q][t] = (unsigned short)sum;
                sum += v;
            }
            up = sum;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int a = __shfl_up(up, off);
                if (lane >= off) up += a;
            }
            if (lane == 63) wsum[w] = up;
        }
        __syncthreads();
        if (t < 256) {
            int b = up - sum;
            for (int q = 0; q < w; q++) b += wsum[q];
            base[t] = b;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < SMALL_ITEMS; r++)
            if (r * 64 < per && w * per + r * 64 + lane < n) {
                const int dg = (key[r] >> (8 * p)) & 255, pos = base[dg] + wc[w][dg] + rank[r];
                lk[pos] = key[r];
                li[pos] = (unsigned short)at[r];
            }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < SMALL_ITEMS; r++) {
            const int i = w * per + r * 64 + lane;
            if (r * 64 < per && i < n) {
                key[r] = lk[i];
                at[r] = li[i];
            }
        }
    }
    int v[SMALL_ITEMS];
#pragma unroll
    for (int r = 0; r < SMALL_ITEMS; r++)
        if (r * 64 < per && w * per + r * 64 + lane < n) v[r] = vals[at[r]];
    __syncthreads();   // every value is read before one is written
#pragma unroll
    for (int r = 0; r < SMALL_ITEMS; r++) {
        const int i = w * per + r * 64 + lane;
        if (r * 64 < per && i < n) {
            keys[i] = key[r];
            vals[i] = v[r];
        }
    }
}

// ------------------------------------------------------------------------
// exclusive scans (device-wide), 2048 elements per 256-thread block
template <class T>
__global__ void __launch_bounds__(BLOCK) k_scan_block(const T* in, T* out, long long n, T* sums, T* total) {
    __shared__ T sh[BLOCK];
    const int t = threadIdx.x;
    long long base = (long long)blockIdx.x * RS_TILE + (long long)t * RS_ITEMS;
    T v[RS_ITEMS];
    T s = 0;
#pragma unroll
    for (int k = 0; k < RS_ITEMS; k++) {
        long long idx = base + k;
        v[k] = idx < n ? in[idx] : (T)0;
        s += v[k];
    }
    sh[t] = s;
    __syncthreads();
    for (int off = 1; off < BLOCK; off <<= 1) {
        T a = t >= off ? sh[t - off] : (T)0;
        __syncthreads();
        sh[t] += a;
        __syncthreads();
    }
    T run = sh[t] - s;
#pragma unroll
    for (int k = 0; k < RS_ITEMS; k++) {
        long long idx = base + k;
        if (idx < n) out[idx] = run;
        run += v[k];
    }
    if (t == BLOCK - 1) {
        sums[blockIdx.x] = sh[t];
        if (total) *total = sh[t];
    }
}
template <class T>
__global__ void __launch_bounds__(BLOCK) k_scan_add(T* out, long long n, const T* offs) {
    long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx < n) out[idx] += offs[idx / RS_TILE];
}

int back_slot(sph_ctx* c) {
    if (!c->back) SPH_HIP(c, hipHostMalloc(&c->back, BACK_BYTES, hipHostMallocDefault));
    return 0;
}
__global__ void k_read_back(const unsigned char* src, unsigned char* dst, int bytes) {
    if ((int)threadIdx.x < bytes) dst[threadIdx.x] = src[threadIdx.x];
}
int read_back(sph_ctx* c, void* dst, const void* src, size_t bytes) {
    if (bytes > BACK_BYTES) return fail(c, SPH_E_ARG, "read_back: too many bytes");
    SPH_TRY(back_slot(c));
    hipLaunchKernelGGL(k_read_back, dim3(1), dim3(BACK_BYTES), 0, c->stream, (const unsigned char*)src,
                       (unsigned char*)c->back, (int)bytes);
    SPH_TRY(launch_check(c, "read_back"));
    SPH_HIP(c, hipStreamSynchronize(c->stream));
    std::memcpy(dst, c->back, bytes);
    return 0;
}

// total: where the last block of sums leaves the total (or null)
template <class T>
static int scan_launches(sph_ctx* c, const T* in, T* out, long long n, T* total) {
    long long nb = (n + RS_TILE - 1) / RS_TILE;
    if (nb < 1) nb = 1;
    T* sums = nullptr;
    T* sums_scan = nullptr;
    SPH_TRY(dalloc(c, &sums, nb + 1));
    hipLaunchKernelGGL(k_scan_block<T>, dim3((unsigned)nb), dim3(BLOCK), 0, c->stream, in, out, n, sums,
                       nb > 1 ? nullptr : total);
    SPH_TRY(launch_check(c, "scan_block"));
    if (nb > 1) {
        SPH_TRY(dalloc(c, &sums_scan, nb + 1));
        SPH_TRY(scan_launches<T>(c, sums, sums_scan, nb, total));
        hipLaunchKernelGGL(k_scan_add<T>, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, out, n, (const T*)sums_scan);
        SPH_TRY(launch_check(c, "scan_add"));
        dfree(c, sums_scan);
    }
    dfree(c, sums);
    return 0;
}
// the total goes to the host (a wait for the stream) only when asked for
template <class T>
static int exclusive_scan(sph_ctx* c, const T* in, T* out, long long n, T* total_out) {
    if (total_out) SPH_TRY(back_slot(c));
    SPH_TRY(scan_launches<T>(c, in, out, n, total_out ? (T*)c->back : nullptr));
    if (total_out) {
        SPH_HIP(c, hipStreamSynchronize(c->stream));
        *total_out = *(const T*)c->back;
    }
    return 0;
}
int exclusive_scan_i32(sph_ctx* c, const int* in, int* out, long long n, int* total) {
    return exclusive_scan<int>(c, in, out, n, total);
}
int exclusive_scan_i64(sph_ctx* c, const long long* in, long long* out, long long n, long long* total) {
    return exclusive_scan<long long>(c, in, out, n, total);
}

// Stable LSD radix sort of (key, value) pairs, keys in [0, max_key]; the
// sorted pairs end in *keys / *vals (the buffers may be swapped with the
// temporaries).
int radix_sort_pairs(sph_ctx* c, int** keys, int** vals, int** ktmp, int** vtmp, int n, int max_key) {
    int bits = 1;
    while ((1LL << bits) <= (long long)max_key) bits++;
    int passes = (bits + 7) / 8;
    if (n <= SMALL_N) {
        SPH_TRY(prof_begin(c, "sort_small", 16.0 * n));
        hipLaunchKernelGGL(k_sort_small, dim3(1), dim3(SMALL_T), 0, c->stream, *keys, *vals, n, passes);
        SPH_TRY(launch_check(c, "sort_small"));
        SPH_TRY(prof_end(c));
        return 0;
    }
    int ntiles = (n + RS_TILE - 1) / RS_TILE;
    int hist_n = 256 * ntiles;
    int* hist = nullptr;
    int* offs = nullptr;
    int* sums = nullptr;
    const int nsums = (hist_n + RS_TILE - 1) / RS_TILE;
    SPH_TRY(dalloc(c, &hist, hist_n));
    SPH_TRY(dalloc(c, &offs, hist_n));
    SPH_TRY(dalloc(c, &sums, nsums));
    int *kin = *keys, *vin = *vals, *kout = *ktmp, *vout = *vtmp;
    for (int p = 0; p < passes; p++) {
        int shift = 8 * p;
        SPH_TRY(prof_begin(c, "radix_hist", 4.0 * n));
        hipLaunchKernelGGL(k_rs_hist, dim3(ntiles), dim3(BLOCK), 0, c->stream, (const int*)kin, n, shift, ntiles, hist);
        SPH_TRY(launch_check(c, "radix_hist"));
        SPH_TRY(prof_end(c));
        hipLaunchKernelGGL(k_scan_block<int>, dim3(nsums), dim3(BLOCK), 0, c->stream, (const int*)hist, offs,
                           (long long)hist_n, sums, (int*)nullptr);
        SPH_TRY(launch_check(c, "scan_block"));
        SPH_TRY(prof_begin(c, "radix_scatter", 16.0 * n));
        hipLaunchKernelGGL(k_rs_scatter, dim3(ntiles), dim3(BLOCK), 0, c->stream, (const int*)kin, (const int*)vin,
                           kout, vout, n, shift, ntiles, (const int*)offs, (const int*)sums, nsums);
        SPH_TRY(launch_check(c, "radix_scatter"));
        SPH_TRY(prof_end(c));
        std::swap(kin, kout);
        std::swap(vin, vout);
    }
    if (kin != *keys) {   // odd pass count: result is in the tmp buffers
        std::swap(*keys, *ktmp);
        std::swap(*vals, *vtmp);
    }
    dfree(c, hist);
    dfree(c, offs);
    dfree(c, sums);
    return 0;
}
static int radix_sort(sph_ctx* c, int max_key) {
    return radix_sort_pairs(c, &c->keys, &c->perm, &c->keys_tmp, &c->perm_tmp, c->n, max_key);
}

// ------------------------------------------------------------------------
// cell start / end, KERNEL_reorder functions_NNPS.cuh:825-838.
// First particle of the sorted order whose key is >= cell, for every cell
// and one past the last: the particles of consecutive cells a..b are
// [cstart[a], cstart[b + 1]), in the order the cells hold them.  A cell's own
// start and end (-1 and 0 where it is empty) are its and the next cell's: a
// block searches CELLS + 1 cells and writes CELLS.  (Two fills, a pass over the
// particles for the bounds and this one took four launches a
// search, 13 us and as much between them; one takes 6.)
constexpr int CELLS = BLOCK - 1;
__global__ void __launch_bounds__(BLOCK) k_cells(int num_cells, const int* keys, int n, int* cstart, int* gstr,
                                                 int* gend) {
    __shared__ int first[BLOCK];
    const int cell = blockIdx.x * CELLS + threadIdx.x;   // 0 .. num_cells + 1
    int lo = 0, hi = cell <= num_cells + 1 ? n : 0;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (keys[mid] < cell) lo = mid + 1;
        else hi = mid;
    }
    first[threadIdx.x] = lo;
    __syncthreads();
    if (threadIdx.x >= CELLS || cell > num_cells + 1) return;
    cstart[cell] = lo;
    if (cell > num_cells) return;
    const int next = first[threadIdx.x + 1];
    gstr[cell] = next > lo ? lo : -1;
    gend[cell] = next > lo ? next : 0;
}

// gather arrays through the permutation, out[f][i] = in[f][perm[i]]: GATHER_N
// arrays a launch (their gathers in flight together, the permutation read
// once).  One array a launch took 58 launches a search: 0.40 ms on the 1 M
// canyon, and 0.14 ms of 3 us launches in each refinement pass of a small case.
// The integers are gathered to scratch by one launch (INTS_OUT) and copied back
// by the next (INTS_BACK).
constexpr int GATHER_N = 16;
enum GatherInts { INTS_NONE, INTS_OUT, INTS_BACK };
struct GatherSet {
    const double* in[GATHER_N];
    double* out[GATHER_N];
    const int* iin[SPH_I_COUNT];
    int* iout[SPH_I_COUNT];
};
template <GatherInts INTS>
__global__ void __launch_bounds__(BLOCK) k_gather(int n, const int* perm, GatherSet G, int nd) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int p = perm[i];
    double v[GATHER_N];
#pragma unroll
    for (int f = 0; f < GATHER_N; f++)
        if (f < nd) v[f] = G.in[f][p];
    if (INTS != INTS_NONE) {
        const int from = INTS == INTS_OUT ? p : i;
        int w[SPH_I_COUNT];
#pragma unroll
        for (int f = 0; f < SPH_I_COUNT; f++) w[f] = G.iin[f][from];
#pragma unroll
        for (int f = 0; f < SPH_I_COUNT; f++) G.iout[f][i] = w[f];
    }
#pragma unroll
    for (int f = 0; f < GATHER_N; f++)
        if (f < nd) G.out[f][i] = v[f];
}

// ------------------------------------------------------------------------
// Neighbour list: the union of the dcell-query window and the binning
// window of particle i (both +-ncell), scanned in increasing cell index so
// entries come out in ascending j, each tagged with the flags of flags.h.
//
// The flags compare the distance r = sqrt(r2) (+- 1e-20) with a radius k.
// Both sides are monotone in r2, so each test is r2 < T with T the least
// double whose root fails it: no root per pair.  T is found per particle
// (k = kappa h, and half of it), and max(T_i, T_j) is the threshold of
// max(h_i, h_j).
struct NLForm {
    int bits;                   // NL_TINY: dp, dm, b differ somewhere (k near 1e-4); NL_VARIES: dp varies
    unsigned long long reach;   // the largest dm, as bits
};
struct NLThr {
    const double *dp, *dm, *b, *bh;   // r + 1e-20 < k; r - 1e-20 < k; r < k; r + 1e-20 < k / 2 (k = kappa h)
    const NLForm* form;
};
constexpr int NL_TINY = 1, NL_VARIES = 2;
// least y >= 0 for which sqrt(y) + add < k does not hold (infinity if none)
__device__ double root_threshold(double k, double add) {
    auto holds = [&](unsigned long long u) { return sqrt(__longlong_as_double((long long)u)) + add < k; };
    const unsigned long long top = 0x7ff0000000000000ull;   // infinity; doubles >= 0 ascend with their bits
    const double y = k > 0.0 ? k * k : 0.0;                 // (NaN: nothing holds, 0)
    unsigned long long u = (unsigned long long)__double_as_longlong(y), lo, hi;
    if (holds(u)) {
        lo = u;
        for (unsigned long long s = 1;; s <<= 1) {
            if (lo == top) return __longlong_as_double((long long)top);
            hi = s < top - lo ? lo + s : top;
            if (!holds(hi)) break;
            lo = hi;
        }
    } else {
        hi = u;
        for (unsigned long long s = 1;; s <<= 1) {
            if (hi == 0) return 0.0;
            lo = hi > s ? hi - s : 0;
            if (holds(lo)) break;
            hi = lo;
        }
    }
    while (hi - lo > 1) {
        const unsigned long long m = lo + (hi - lo) / 2;
        if (holds(m)) lo = m;
        else hi = m;
    }
    return __longlong_as_double((long long)hi);
}
__global__ void __launch_bounds__(BLOCK) k_nl_thresholds(int n, const double* h, double kappa, double* dp, double* dm,
                                                         double* b, double* bh, NLForm* form) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    int fm = 0;
    unsigned long long far = 0;
    if (i < n) {
        const double k = kappa * h[i];
        const double tp = root_threshold(k, 1e-20), tm = root_threshold(k, -1e-20), t0 = root_threshold(k, 0.0);
        dp[i] = tp;
        dm[i] = tm;
        b[i] = t0;
        bh[i] = root_threshold(kappa * (0.5 * h[i]), 1e-20);
        far = (unsigned long long)__double_as_longlong(tm);
        fm = (tp != tm || tp != t0 ? NL_TINY : 0) | (h[i] != h[0] ? NL_VARIES : 0);
    }
    for (int bit = 1; bit <= NL_VARIES; bit <<= 1)
        if (__ballot(fm & bit) && (threadIdx.x & 63) == 0 && !(form->bits & bit)) atomicOr(&form->bits, bit);
    for (int off = 32; off > 0; off >>= 1) far = max(far, (unsigned long long)__shfl_xor((long long)far, off, 64));
    if ((threadIdx.x & 63) == 0 && far > form->reach) atomicMax(&form->reach, far);
}
// Where the particles of a cell can lie along an axis: its share of the
// binning range, `pad` wider for the float arithmetic here and in the binning
// (together below 1e-6 of the range and of a coordinate), and without end
// beyond the first and the last cell, which take what lies outside.
struct Axis {
    float lo, w, inv, pad;
    int N;
    __device__ Axis(float mn, float mx, int n)
        : lo(mn), w((mx - mn) / (float)n), inv(1.0f / w), pad(4e-6f * (fabsf(mn) + fabsf(mx))), N(n) {}
    // distance of cell c to [a, b], never too large
    __device__ float gap(int c, float a, float b) const {
        const float below = c < N - 1 ? a - (lo + (float)(c + 1) * w + pad) : 0.0f;
        const float above = c > 0 ? (lo + (float)c * w - pad) - b : 0.0f;
        return fmaxf(fmaxf(below, above), 0.0f);
    }
    // the cell that holds v (a NaN, of an axis without extent: the first)
    __device__ int cell(float v) const { return (int)fminf(fmaxf(floorf((v - lo) * inv), 0.0f), (float)(N - 1)); }
};
// One 64-lane wave lists NL_P consecutive particles, those of one window
// together: the window's x-rows are numbered z-major then y (lane k describes
// row k of a batch of 64), their particle ranges are flattened into one
// candidate order v, each round of 64 candidates is loaded once for the
// particles that share it, and compacted in order with a ballot per
// particle, so the lists are the ones a serial scan in cell order produces.
// Bound by vector instructions, in equal parts of a window's set-up and of
// its candidates.  A wave a particle, with a root a pair, a six-step search
// for each candidate's row and no row left out, took 1365 of them a particle
// and 2.85 ms for 1 M particles of ~590 candidates and 99 entries; this takes
// 1.43 ms (count alone 2.5 -> 1.1 ms).
constexpr int NL_P = 4;
static_assert(SLICE % NL_P == 0, "a wave's particles share a slice");
// inclusive prefix sum over the wave's lanes
__device__ __forceinline__ int wave_incl(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1, 2, 4, 8: rows of 16 lanes
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);   // row_bcast:15 into rows 1, 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);   // row_bcast:31 into rows 2, 3
    return v;
}
template <bool FILL, bool TINY, bool VARIES>
__device__ __forceinline__ int nl_wave(int i0, int np, const Grid& g, const double* x, const double* y,
                                        const double* z, const NLThr& t, const int* ncell, int* marks, unsigned* out,
                                        int cap, int* cnt) {
    const int lane = threadIdx.x & 63;
    int longest = 0;
    const sph_domain& d = g.d;
    // lane p: the cells of particle i0 + p
    const int ip = i0 + min(lane, np - 1);
    const double xp = x[ip], yp = y[ip], zp = z[ip], dpp = t.dp[ip], bhp = t.bh[ip];
    const Cell qp = query_cell(d, xp, yp, zp), bp = bin_cell(d, xp, yp, zp);
    const int ncp = ncell[ip];
    const double dmp = TINY ? t.dm[ip] : 0.0, tbp = TINY ? t.b[ip] : 0.0;
    auto at64 = [](double v, int l) {   // lane l's value, wave-uniform
        const long long u = __double_as_longlong(v);
        const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)u, l);
        const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(u >> 32), l);
        return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
    };
    // no pair of r2 >= reach has a flag
    const float reach = (float)__longlong_as_double((long long)t.form->reach);
    const Axis ax(d.x_min, d.x_max, d.NI), ay(d.y_min, d.y_max, d.NJ), az(d.z_min, d.z_max, d.NK);
    for (int a = 0; a < np;) {
        auto at = [&](int v) { return __builtin_amdgcn_readlane(v, a); };
        const Cell q{at(qp.i), at(qp.j), at(qp.k)}, b{at(bp.i), at(bp.j), at(bp.k)};
        const int nc = at(ncp);
        const unsigned long long same =
            __ballot(qp.i == q.i && qp.j == q.j && qp.k == q.k && bp.i == b.i && bp.j == b.j && bp.k == b.k && ncp == nc);
        int C = 1;   // particles a .. a + C - 1 share the window
        while (a + C < np && ((same >> (a + C)) & 1ULL)) C++;
        double xi[NL_P], yi[NL_P], zi[NL_P], dp[NL_P], dm[NL_P], tb[NL_P], th[NL_P];
        int m[NL_P] = {};
        float bx0 = 0, bx1 = 0, by0 = 0, by1 = 0, bz0 = 0, bz1 = 0;   // the particles' box
#pragma unroll
        for (int p = 0; p < NL_P; p++) {
            if (p >= C) break;
            const int l = a + p;
            xi[p] = at64(xp, l); yi[p] = at64(yp, l); zi[p] = at64(zp, l);
            dp[p] = at64(dpp, l); th[p] = at64(bhp, l);
            dm[p] = TINY ? at64(dmp, l) : 0.0; tb[p] = TINY ? at64(tbp, l) : 0.0;
            const float fx = (float)xi[p], fy = (float)yi[p], fz = (float)zi[p];
            bx0 = p ? fminf(bx0, fx) : fx; bx1 = p ? fmaxf(bx1, fx) : fx;
            by0 = p ? fminf(by0, fy) : fy; by1 = p ? fmaxf(by1, fy) : fy;
            bz0 = p ? fminf(bz0, fz) : fz; bz1 = p ? fmaxf(bz1, fz) : fz;
        }
        const bool one = q.i == b.i && q.j == b.j && q.k == b.k;   // the two windows are one
        const int jlo = max(min(q.j, b.j) - nc, 0), jhi = min(max(q.j, b.j) + nc, d.NJ - 1);
        const int klo = max(min(q.k, b.k) - nc, 0), khi = min(max(q.k, b.k) + nc, d.NK - 1);
        const int nj = max(jhi - jlo + 1, 0), nk = max(khi - klo + 1, 0), nrows = nj * nk;
        for (int r0 = 0; r0 < nrows; r0 += 64) {
            // lane k: row r0 + k of the union window
            int rs = 0, rl = 0, base = 0, flags = 0;
            const int rk = r0 + lane;
            if (rk < nrows) {
                const int ck = klo + rk / nj, cj = jlo + rk % nj;
                const bool rowD = abs(cj - q.j) <= nc && abs(ck - q.k) <= nc;
                const bool rowB = abs(cj - b.j) <= nc && abs(ck - b.k) <= nc;
                int c0 = INT_MAX, c1 = INT_MIN;
                if (rowD) { c0 = min(c0, q.i - nc); c1 = max(c1, q.i + nc); }
                if (rowB) { c0 = min(c0, b.i - nc); c1 = max(c1, b.i + nc); }
                const float gy = ay.gap(cj, by0, by1), gz = az.gap(ck, bz0, bz1), left = reach - gy * gy - gz * gz;
                if (left < -1e-5f * reach) c1 = INT_MIN;   // the row is out of reach
                const float half = sqrtf(fmaxf(left, 0.0f) + 2e-5f * reach);
                c0 = max(max(c0, 0), ax.cell(bx0 - half - ax.pad));
                c1 = min(min(c1, d.NI - 1), ax.cell(bx1 + half + ax.pad));
                base = d.NI * cj + d.NI * d.NJ * ck;
                flags = (rowD ? 1 : 0) | (rowB ? 2 : 0);
                if ((rowD || rowB) && c0 <= c1) {
                    rs = g.cstart[base + c0];
                    rl = g.cstart[base + c1 + 1] - rs;
                }
            }
            const int incl = wave_incl(rl);
            const int excl = incl - rl, total = __builtin_amdgcn_readlane(incl, 63), first = rs - excl;
            int held = 0;   // the row that holds the last candidate of the round before
            for (int v0 = 0; v0 < total; v0 += 64) {
                // the row of candidate v: each row that starts in the round marks its first candidate
                marks[lane] = -1;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (rl > 0 && excl >= v0 && excl < v0 + 64) marks[excl - v0] = lane;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const int mk = marks[lane];
                const unsigned long long M = __ballot(mk >= 0), upto = M & (~0ULL >> (63 - lane));
                const int near = __shfl(mk, upto ? 63 - __clzll((long long)upto) : 0, 64);
                const int row = upto ? near : held;
                if (M) held = __builtin_amdgcn_readlane(mk, 63 - __clzll((long long)M));
                const int v = min(v0 + lane, total - 1);
                const int rowv = v0 + lane < total ? row : held;
                const int j = __shfl(first, rowv, 64) + v;
                bool inD = v0 + lane < total, inB = inD;
                if (!one) {
                    const int rflags = __shfl(flags, rowv, 64);
                    inD = inD && (rflags & 1);
                    inB = inB && (rflags & 2);
                    if (q.i != b.i) {
                        const int ci = g.keys[j] - __shfl(base, rowv, 64);
                        inD = inD && abs(ci - q.i) <= nc;
                        inB = inB && abs(ci - b.i) <= nc;
                    }
                }
                const double xj = x[j], yj = y[j], zj = z[j];
                const double dpj = VARIES ? t.dp[j] : 0.0, dmj = VARIES && TINY ? t.dm[j] : 0.0;
#pragma unroll
                for (int p = 0; p < NL_P; p++) {
                    if (p >= C) break;
                    const double r2 =
                        (xi[p] - xj) * (xi[p] - xj) + (yi[p] - yj) * (yi[p] - yj) + (zi[p] - zj) * (zi[p] - zj);
                    const double kd = VARIES ? fmax(dp[p], dpj) : dp[p];
                    unsigned f = 0;
                    if (TINY) {
                        const double km = VARIES ? fmax(dm[p], dmj) : dm[p];
                        if (inD)
                            f = (r2 < kd ? F_DP : 0u) | (r2 < km ? F_DM : 0u) | (r2 < dp[p] ? F_HP : 0u) |
                                (r2 < dm[p] ? F_HM : 0u);
                        if (inB) f |= (r2 > 0.0 && r2 < tb[p] ? F_B : 0u) | (r2 < th[p] ? F_BH : 0u);
                    } else {
                        const bool own = r2 < dp[p];
                        if (inD) f = (r2 < kd ? F_DP | F_DM : 0u) | (own ? F_HP | F_HM : 0u);
                        if (inB) f |= (r2 > 0.0 && own ? F_B : 0u) | (r2 < th[p] ? F_BH : 0u);
                    }
                    const unsigned long long hit = __ballot(f != 0);
                    if (FILL && f) {
                        const int slot = m[p] + (int)__builtin_amdgcn_mbcnt_hi(
                                                    (unsigned)(hit >> 32),
                                                    __builtin_amdgcn_mbcnt_lo((unsigned)hit, 0u));
                        if (slot < cap) out[(size_t)slot * SLICE + a + p] = (unsigned)j | f;
                    }
                    m[p] += __popcll(hit);
                }
            }
        }
        if (lane < C) {
            int v = 0;
#pragma unroll
            for (int p = 0; p < NL_P; p++) v = lane == p ? m[p] : v;
            cnt[a + lane] = v;
        }
#pragma unroll
        for (int p = 0; p < NL_P; p++) longest = max(longest, m[p]);
        a += C;
    }
    return longest;
}
// the first particle of this wave.  xcd_block: a list slice's 64 particles on
// one XCD, so their interleaved entries fill whole lines in one L2
__device__ __forceinline__ int nl_first() {
    return __builtin_amdgcn_readfirstlane(
        (int)((((long long)xcd_block() * blockDim.x + threadIdx.x) >> 6) * NL_P));
}
template <bool FILL>
__device__ __forceinline__ int nl_lists(int i0, int np, const Grid& g, const double* x, const double* y,
                                        const double* z, const NLThr& t, const int* ncell, int* marks, unsigned* out,
                                        int cap, int* cnt) {
    const int form = __builtin_amdgcn_readfirstlane(t.form->bits);
    if (form & NL_TINY) return nl_wave<FILL, true, true>(i0, np, g, x, y, z, t, ncell, marks, out, cap, cnt);
    if (form & NL_VARIES) return nl_wave<FILL, false, true>(i0, np, g, x, y, z, t, ncell, marks, out, cap, cnt);
    return nl_wave<FILL, false, false>(i0, np, g, x, y, z, t, ncell, marks, out, cap, cnt);
}
__global__ void __launch_bounds__(BLOCK) k_nl_count(int n, Grid g, const double* x, const double* y, const double* z,
                                                    NLThr t, const int* ncell, int* cnt) {
    __shared__ int marks[BLOCK];
    const int i0 = nl_first();
    if (i0 >= n) return;   // whole waves
    nl_lists<false>(i0, min(NL_P, n - i0), g, x, y, z, t, ncell, marks + (threadIdx.x & ~63), nullptr, 0, cnt + i0);
}
// fill pass; with over (a fill without a count pass) into the room of each
// slice, over = 1 when a list does not fit
__global__ void __launch_bounds__(BLOCK) k_nl_fill(int n, Grid g, const double* x, const double* y, const double* z,
                                                   NLThr t, const int* ncell, const long long* slice_off,
                                                   long long total, unsigned* ent, int* cnt, int* over) {
    __shared__ int marks[BLOCK];
    const int i0 = nl_first();
    if (i0 >= n) return;   // whole waves
    const int s = i0 >> 6, np = min(NL_P, n - i0);
    const long long end = s + 1 < (n + SLICE - 1) / SLICE ? slice_off[s + 1] : total;
    const int cap = (int)((end - slice_off[s]) / SLICE);
    const int longest = nl_lists<true>(i0, np, g, x, y, z, t, ncell, marks + (threadIdx.x & ~63),
                                      ent + slice_off[s] + (i0 & 63), cap, cnt + i0);
    if (over && longest > cap) over[0] = 1;
}
// room of each slice for a fill without a count pass
__global__ void __launch_bounds__(BLOCK) k_slice_spare(int nslices, const long long* prev, long long spare,
                                                       long long* w) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nslices) w[s] = prev[s] + spare * SLICE;
}
__global__ void __launch_bounds__(BLOCK) k_slice_width(int n, int nslices, const int* cnt, long long* w) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nslices) return;
    int m = 0;
    for (int l = 0; l < SLICE; l++) {
        int i = s * SLICE + l;
        if (i < n) m = max(m, cnt[i]);
    }
    w[s] = (long long)m * SLICE;
}

// ------------------------------------------------------------------------
static int permute_state(sph_ctx* c) {
    const int n = c->n;
    std::vector<double**> arr;
    for (int f = 0; f < SPH_F_COUNT_F64 + 3; f++)
        if (c->pf[f]) arr.push_back(&c->pf[f]);
    for (int f = 0; f < 10; f++) arr.push_back(&c->p2[f]);
    for (int f = 15; f < 18; f++) arr.push_back(&c->q[f]);
    if (c->apr_target) arr.push_back(&c->apr_target);
    // Each state array is swapped for its gathered copy.  The copies go to the
    // working copies' arrays, of the context's capacity like all state arrays
    // (refinement appends particles past n): nothing reads those between a
    // step's end and the next one's start, which writes them all.  (Blocks of
    // its own took a search 152 bytes a particle, which stayed in the cache.)
    static_assert(MF_COUNT >= GATHER_N + (SPH_I_COUNT + 1) / 2, "room for the copies");
    int* itmp[SPH_I_COUNT];
    for (int f = 0; f < SPH_I_COUNT; f++) itmp[f] = (int*)c->sm[GATHER_N + f / 2] + (size_t)(f % 2) * c->cap;
    SPH_TRY(prof_begin(c, "permute", 0));
    const size_t launches = std::max<size_t>(2, (arr.size() + GATHER_N - 1) / GATHER_N);
    for (size_t l = 0; l < launches; l++) {
        const size_t a0 = std::min(arr.size(), l * GATHER_N);
        const int nd = (int)std::min<size_t>(GATHER_N, arr.size() - a0);
        GatherSet G{};
        for (int f = 0; f < nd; f++) {
            G.in[f] = *arr[a0 + f];
            G.out[f] = c->sm[f];
        }
        for (int f = 0; f < SPH_I_COUNT; f++) {
            G.iin[f] = l == 0 ? c->pi[f] : itmp[f];
            G.iout[f] = l == 0 ? itmp[f] : c->pi[f];
        }
        auto* const kern = l == 0 ? k_gather<INTS_OUT> : l == 1 ? k_gather<INTS_BACK> : k_gather<INTS_NONE>;
        hipLaunchKernelGGL(kern, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, (const int*)c->perm, G, nd);
        SPH_TRY(launch_check(c, "permute"));
        for (int f = 0; f < nd; f++) std::swap(*arr[a0 + f], c->sm[f]);
    }
    SPH_TRY(prof_end(c));
    return 0;
}

// Order of the record-gathering particle passes (thread -> particle):
// particles with lists of at most NL_HEAVY entries first, in their order,
// then the longer ones (coarse particles beside refined zones), so that
// those do not hold waves of short lists for their length.  Null when no
// list is that long.  A pass computes each particle on its own, so the
// order changes no result.
constexpr int NL_HEAVY = 512;
__global__ void __launch_bounds__(BLOCK) k_heavy_flag(int n, const int* cnt, int* flag) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flag[i] = cnt[i] > NL_HEAVY ? 1 : 0;
}
__global__ void __launch_bounds__(BLOCK) k_porder(int n, int nlight, const int* flag, const int* scan, int* order) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    order[flag[i] ? nlight + scan[i] : i - scan[i]] = i;
}
static int build_porder(sph_ctx* c) {
    const int n = c->n;
    dfree(c, c->porder);
    c->porder = nullptr;
    c->n_heavy = 0;
    if (n == 0) return 0;
    int *flag = nullptr, *scan = nullptr;
    SPH_TRY(dalloc(c, &flag, n));
    SPH_TRY(dalloc(c, &scan, n));
    hipLaunchKernelGGL(k_heavy_flag, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, (const int*)c->nl_cnt, flag);
    SPH_TRY(launch_check(c, "porder"));
    int nheavy = 0;
    SPH_TRY(exclusive_scan_i32(c, flag, scan, n, &nheavy));
    c->n_heavy = nheavy;
    if (nheavy > 0) {
        SPH_TRY(dalloc(c, &c->porder, n));
        hipLaunchKernelGGL(k_porder, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, n - nheavy, (const int*)flag,
                           (const int*)scan, c->porder);
        SPH_TRY(launch_check(c, "porder"));
    }
    dfree(c, flag);
    dfree(c, scan);
    return 0;
}

// The list of a search.  When the previous search
// had as many slices (the particles keep their cell order, and move little
// between searches), the fill runs at once into each slice's previous
// width plus NL_SPARE entries; if a list does not fit, the search counts
// first and fills slices of exact widths.  The entries are the same either
// way.
constexpr int NL_SPARE = 8;
static int build_neighbor_list(sph_ctx* c) {
    const int n = c->n;
    int nslices = (n + SLICE - 1) / SLICE;
    dfree(c, c->nl_cnt); c->nl_cnt = nullptr;
    dfree(c, c->nl_slice_off); c->nl_slice_off = nullptr;
    dfree(c, c->nl_ent); c->nl_ent = nullptr;
    SPH_TRY(dalloc(c, &c->nl_cnt, n));
    SPH_TRY(dalloc(c, &c->nl_slice_off, nslices + 1));
    Grid g = c->grid();
    const double *x = c->pf[SPH_F_X], *y = c->pf[SPH_F_Y], *z = c->pf[SPH_F_Z], *h = c->pf[SPH_F_H];
    const unsigned nlgrid = (unsigned)grid1(((long long)n + NL_P - 1) / NL_P * 64);
    double* const* const thr = c->sm;   // four arrays of the working copies (see permute_state)
    NLForm* form = nullptr;
    SPH_TRY(dalloc(c, &form, 1));
    SPH_HIP(c, hipMemsetAsync(form, 0, sizeof(NLForm), c->stream));
    const NLThr t{thr[0], thr[1], thr[2], thr[3], form};
    SPH_TRY(prof_begin(c, "nl_thresholds", 40.0 * n));
    hipLaunchKernelGGL(k_nl_thresholds, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, h, c->prm.kappa, thr[0], thr[1],
                       thr[2], thr[3], form);
    SPH_TRY(launch_check(c, "nl_thresholds"));
    SPH_TRY(prof_end(c));
    long long* w = nullptr;
    SPH_TRY(dalloc(c, &w, nslices + 1));
    long long total = 0;
    if (c->nl_wprev && c->nl_wprev_n == nslices) {
        int* over = nullptr;
        SPH_TRY(dalloc(c, &over, 1));
        SPH_HIP(c, hipMemsetAsync(over, 0, sizeof(int), c->stream));
        hipLaunchKernelGGL(k_slice_spare, dim3(grid1(nslices)), dim3(BLOCK), 0, c->stream, nslices,
                           (const long long*)c->nl_wprev, (long long)NL_SPARE, w);
        SPH_TRY(launch_check(c, "slice_width"));
        SPH_TRY(exclusive_scan_i64(c, w, c->nl_slice_off, nslices, &total));
        SPH_TRY(dalloc(c, &c->nl_ent, (size_t)total + 1));
        SPH_TRY(prof_begin(c, "nl_fill", 0));
        hipLaunchKernelGGL(k_nl_fill, dim3(nlgrid), dim3(BLOCK), 0, c->stream, n, g, x, y, z, t,
                           (const int*)c->pi[SPH_I_NCELL], (const long long*)c->nl_slice_off, total,
                           c->nl_ent, c->nl_cnt, over);
        SPH_TRY(launch_check(c, "nl_fill"));
        SPH_TRY(prof_end(c));
        int h_over = 0;
        SPH_TRY(read_back(c, &h_over, over, sizeof(int)));
        dfree(c, over);
        if (!h_over) {
            // exact widths of this search: the next one's guess
            hipLaunchKernelGGL(k_slice_width, dim3(grid1(nslices)), dim3(BLOCK), 0, c->stream, n, nslices,
                               (const int*)c->nl_cnt, c->nl_wprev);
            SPH_TRY(launch_check(c, "slice_width"));
            c->nl_total = total;
            dfree(c, w);
            dfree(c, form);
            return build_porder(c);
        }
        dfree(c, c->nl_ent);
        c->nl_ent = nullptr;
    }
    SPH_TRY(prof_begin(c, "nl_count", 0));
    hipLaunchKernelGGL(k_nl_count, dim3(nlgrid), dim3(BLOCK), 0, c->stream, n, g, x, y, z, t,
                       (const int*)c->pi[SPH_I_NCELL], c->nl_cnt);
    SPH_TRY(launch_check(c, "nl_count"));
    SPH_TRY(prof_end(c));
    hipLaunchKernelGGL(k_slice_width, dim3(grid1(nslices)), dim3(BLOCK), 0, c->stream, n, nslices,
                       (const int*)c->nl_cnt, w);
    SPH_TRY(launch_check(c, "slice_width"));
    if (c->nl_wprev_n != nslices) {
        dfree(c, c->nl_wprev);
        c->nl_wprev = nullptr;
        SPH_TRY(dalloc(c, &c->nl_wprev, nslices + 1));
        c->nl_wprev_n = nslices;
    }
    SPH_HIP(c, hipMemcpyAsync(c->nl_wprev, w, sizeof(long long) * nslices, hipMemcpyDeviceToDevice, c->stream));
    SPH_TRY(exclusive_scan_i64(c, w, c->nl_slice_off, nslices, &total));
    dfree(c, w);
    c->nl_total = total;
    SPH_TRY(dalloc(c, &c->nl_ent, (size_t)total + 1));
    SPH_TRY(prof_begin(c, "nl_fill", 0));
    hipLaunchKernelGGL(k_nl_fill, dim3(nlgrid), dim3(BLOCK), 0, c->stream, n, g, x, y, z, t,
                       (const int*)c->pi[SPH_I_NCELL], (const long long*)c->nl_slice_off, total, c->nl_ent,
                       c->nl_cnt, (int*)nullptr);
    SPH_TRY(launch_check(c, "nl_fill"));
    SPH_TRY(prof_end(c));
    dfree(c, form);
    return build_porder(c);
}

// The particles the Neumann pass updates (every p_type but fluid), in the
// sorted order of the search.
__global__ void __launch_bounds__(BLOCK) k_nm_flag(int n, const int* p_type, int* flag) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flag[i] = p_type[i] != 1 ? 1 : 0;
}
__global__ void __launch_bounds__(BLOCK) k_nm_fill(int n, const int* flag, const int* scan, int* list) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && flag[i]) list[scan[i]] = i;
}
static int neumann_list(sph_ctx* c) {
    const int n = c->n;
    int *flag = nullptr, *scan = nullptr, cnt = 0;
    SPH_TRY(dalloc(c, &flag, n));
    SPH_TRY(dalloc(c, &scan, n));
    hipLaunchKernelGGL(k_nm_flag, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, (const int*)c->pi[SPH_I_P_TYPE], flag);
    SPH_TRY(launch_check(c, "nm_flag"));
    SPH_TRY(exclusive_scan_i32(c, flag, scan, n, &cnt));
    dfree(c, c->nm_list);
    c->nm_list = nullptr;
    SPH_TRY(dalloc(c, &c->nm_list, cnt > 0 ? cnt : 1));
    hipLaunchKernelGGL(k_nm_fill, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, (const int*)flag, (const int*)scan,
                       c->nm_list);
    SPH_TRY(launch_check(c, "nm_fill"));
    c->nm_count = cnt;
    dfree(c, flag);
    dfree(c, scan);
    return 0;
}

// The neighbour list (and the list of the Neumann pass's particles) alone, on
// the cells and order of the last search.
int nnps_list(sph_ctx* c) {
    SPH_TRY(neumann_list(c));
    return build_neighbor_list(c);
}

// Full count==0 search on the current persistent state (any order): cell
// keys, stable sort, cell bounds, permutation of the state and, when
// build_list, the per-particle neighbour list.
int nnps_run(sph_ctx* c, bool build_list) {
    const int n = c->n;
    const sph_domain& d = c->dom;
    if (!c->keys) {
        // sized for the context's capacity: refinement adds particles
        SPH_TRY(dalloc(c, &c->keys, c->cap));
        SPH_TRY(dalloc(c, &c->perm, c->cap));
        SPH_TRY(dalloc(c, &c->keys_tmp, c->cap));
        SPH_TRY(dalloc(c, &c->perm_tmp, c->cap));
    }
    if (!c->gstr) {
        SPH_TRY(dalloc(c, &c->gstr, (size_t)d.num_cells + 1));
        SPH_TRY(dalloc(c, &c->gend, (size_t)d.num_cells + 1));
        SPH_TRY(dalloc(c, &c->cstart, (size_t)d.num_cells + 2));
    }
    SPH_TRY(prof_begin(c, "hash", (3.0 * 8 + 4 + 8) * n));
    hipLaunchKernelGGL(k_hash, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, d, (const int*)c->pi[SPH_I_I_TYPE],
                       (const double*)c->pf[SPH_F_X], (const double*)c->pf[SPH_F_Y], (const double*)c->pf[SPH_F_Z],
                       c->keys, c->perm);
    SPH_TRY(launch_check(c, "hash"));
    SPH_TRY(prof_end(c));
    SPH_TRY(radix_sort(c, d.num_cells));
    SPH_TRY(prof_begin(c, "cell_bounds", 4.0 * n + 8.0 * (d.num_cells + 1)));
    hipLaunchKernelGGL(k_cells, dim3((unsigned)(((long long)d.num_cells + 2 + CELLS - 1) / CELLS)), dim3(BLOCK), 0,
                       c->stream, d.num_cells, (const int*)c->keys, n, c->cstart, c->gstr, c->gend);
    SPH_TRY(launch_check(c, "cells"));
    SPH_TRY(prof_end(c));
    SPH_TRY(permute_state(c));
    if (build_list) SPH_TRY(nnps_list(c));
    c->searched = true;
    c->generation++;   // state arrays were swapped for their sorted copies
    return 0;
}

int set_ncell_run(sph_ctx* c) {
    const int n = c->n;
    hipLaunchKernelGGL(k_set_ncell, dim3(grid1(n)), dim3(BLOCK), 0, c->stream, n, (const int*)c->pi[SPH_I_I_TYPE],
                       (const double*)c->pf[SPH_F_H], (const double*)c->pf[SPH_F_COUNT_F64 + 2],
                       c->pi[SPH_I_NCELL]);
    return launch_check(c, "set_ncell");
}

}  // namespace sph
