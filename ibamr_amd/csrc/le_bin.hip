// le_bin.hip -- point binning: IndexUtilities::getCellIndex per point (FP64, bit-exact,
// IndexUtilities-inl.h:52-72, level form :226-243), then a stable LSD radix sort of
// the points by spread bin (no device-wide atomics) and CSR bin offsets.
#include "le_plan_internal.h"

namespace ibamr
{
namespace
{
struct BinArgs
{
    const double* X;
    int n;
    double xlo[3], xhi[3], dx[3];
    int ref_lo[3], ref_hi[3];
    int sel_lo[3], sel_hi[3];
    int dom_lo[3], dom_hi[3];
    int nb[3];
    int nsb[3];
    int bin;
    int nmem;
    int ksub;   // bits of the plane-in-bin part of a key (0: bins only)
    int* nactive;  // cleared for k_bin_bounds (null: not counted)
    int* keys;
    int4* cell;  // getCellIndex of every point, in the caller's order
};

// IndexUtilities::getCellIndex (IndexUtilities-inl.h:52-72) on the level domain
// (level overload :226-243), then the spread bin of the cell.
template <int NDIM>
__global__ void k_bin_keys(BinArgs a)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p == 0 && a.nactive) *a.nactive = 0;
    if (p >= a.n) return;
    int c[3] = {0, 0, 0};
    int raw[3] = {0, 0, 0};
    bool inside = true;
#pragma unroll
    for (int d = 0; d < NDIM; ++d)
    {
        const double v = cell_index_d(a.X[NDIM * p + d], a.xlo[d], a.xhi[d], a.dx[d], a.ref_lo[d], a.ref_hi[d]);
        // NaN or far outside: not selected
        inside = inside && (v >= (double)a.sel_lo[d]) && (v <= (double)a.sel_hi[d]);
        c[d] = inside ? (int)v : a.dom_lo[d];
        // the index itself where an int holds it (INT_MIN for NaN or beyond 2^30)
        raw[d] = (v >= -1073741824.0 && v <= 1073741824.0) ? (int)v : INT_MIN;
    }
    int key = a.nmem << a.ksub;  // sentinel: sorts after every bin
    if (inside)
    {
        // bin, then the cell's plane inside the bin along the last axis (z in
        // 3-D, y in 2-D), so that a bin's points are sorted by plane whatever the
        // input order and a 64-point chunk of a crowded bin spans few z planes
        int b[3] = {0, 0, 0};
#pragma unroll
        for (int d = 0; d < NDIM; ++d) b[d] = (c[d] - a.dom_lo[d]) / a.bin;
        const int l = c[NDIM - 1] - a.dom_lo[NDIM - 1] - b[NDIM - 1] * a.bin;
        key = (bin_mem(NDIM, b[0], b[1], b[2], a.nb, a.nsb) << a.ksub) | (a.ksub ? l : 0);
    }
    a.keys[p] = key;
    a.cell[p] = make_int4(raw[0], raw[1], raw[2], 0);
}

// Stable LSD radix sort of the bin keys, carrying the point indices: after it
// the points are grouped by bin and, inside a bin, in index order, so every
// later kernel sees one deterministic order.  Device-wide atomics are avoided
// (on a multi-XCD GPU they are resolved past the per-XCD L2): per pass, a
// block histogram in LDS, an exclusive scan of each digit's block counts, and a
// scatter that adds up the digits' totals and ranks equal digits with wave ballots.
//
// At a few million keys a pass is bound by latency, not by its bytes: there are
// only two or so workgroups per CU.  So each thread holds its keys in registers
// (all loads in flight at once), each wavefront ranks its own run of consecutive
// keys without a barrier, and the tile is put in digit order in LDS, so that the
// stores of a digit's keys are consecutive.  2 M keys of
// 20 bits: 2 x (11 + 5 + 17) us; 3 x (7 + 15 + 21) us with 8-bit digits, a scan
// over all counts in three kernels, and a scatter of three barriers per 256 keys.
// (Kernel by kernel an 8-bit digit is cheaper, 5 + 5 + 15 us: wide digits are taken
// only where they save a pass.)

// hist[d * nblocks + block] = number of keys of this block's tile with digit d
template <int BITS>
__global__ __launch_bounds__(RS_THREADS) void k_rs_hist(const int* __restrict__ keys, int n, int shift,
                                                        int nblocks, int* __restrict__ hist)
{
    constexpr int D = 1 << BITS;
    __shared__ int s_cnt[D];
    const int t = threadIdx.x;
    for (int d = t; d < D; d += RS_THREADS) s_cnt[d] = 0;
    const int i0 = blockIdx.x * RS_TILE;
    int key[RS_ROUNDS];
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r)
    {
        const int i = i0 + r * RS_THREADS + t;
        key[r] = i < n ? keys[i] : -1;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r)
        if (key[r] >= 0) atomicAdd(&s_cnt[(key[r] >> shift) & (D - 1)], 1);  // LDS: exact, order free
    __syncthreads();
    for (int d = t; d < D; d += RS_THREADS) hist[(size_t)d * nblocks + blockIdx.x] = s_cnt[d];
}

__device__ __forceinline__ int wave_inclusive_sum(int v, int lane)
{
#pragma unroll
    for (int o = 1; o < 64; o <<= 1)
    {
        const int u = __shfl_up(v, o);
        if (lane >= o) v += u;
    }
    return v;
}

// off[d * nblocks + b] = keys of digit d in the blocks before b; total[d] = keys of
// digit d.  One workgroup per digit.
__global__ __launch_bounds__(256) void k_rs_scan(const int* __restrict__ hist, int nblocks, int* __restrict__ off,
                                                 int* __restrict__ total)
{
    __shared__ int s_w[4];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const size_t row = (size_t)blockIdx.x * nblocks;
    int run = 0;
    for (int b0 = 0; b0 < nblocks; b0 += 256)
    {
        const int b = b0 + t;
        const int v = b < nblocks ? hist[row + b] : 0;
        const int inc = wave_inclusive_sum(v, lane);
        if (lane == 63) s_w[wv] = inc;
        __syncthreads();
        int before = run, all = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w)
        {
            before += w < wv ? s_w[w] : 0;
            all += s_w[w];
        }
        if (b < nblocks) off[row + b] = before + inc - v;
        run += all;
        __syncthreads();
    }
    if (t == 0) total[blockIdx.x] = run;
}

// Orders the LDS accesses of a wavefront's lanes before and after it.
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Block b's keys of digit d go to (keys of smaller digits) + off[d * nblocks + b]
// onward, in tile order.  vals_in == nullptr: the value of element i is i (first pass).
template <int BITS>
__global__ __launch_bounds__(RS_THREADS) void k_rs_scatter(const int* __restrict__ keys_in,
                                                           const int* __restrict__ vals_in, int n, int shift,
                                                           int nblocks, const int* __restrict__ off,
                                                           const int* __restrict__ total,
                                                           int* __restrict__ keys_out, int* __restrict__ vals_out)
{
    constexpr int D = 1 << BITS;
    constexpr int DPT = D > RS_THREADS ? D / RS_THREADS : 1;  // consecutive digits of a thread
    __shared__ unsigned short s_wc[RS_WAVES][D];  // a wavefront's keys per digit, then where they start in the tile
    __shared__ int s_gofs[D];                     // output position minus position in the tile
    __shared__ int s_key[RS_TILE], s_val[RS_TILE];
    __shared__ int s_wt[RS_WAVES], s_wl[RS_WAVES];
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int i0 = blockIdx.x * RS_TILE;
    const int iw = i0 + wv * (64 * RS_ROUNDS) + lane;  // a wavefront's keys are consecutive
    int key[RS_ROUNDS], val[RS_ROUNDS], rank[RS_ROUNDS];
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r)
    {
        const int i = iw + r * 64;
        key[r] = i < n ? keys_in[i] : -1;
        val[r] = i < n ? (vals_in ? vals_in[i] : i) : 0;
    }
    int gtot[DPT], goff[DPT];
#pragma unroll
    for (int k = 0; k < DPT; ++k)
    {
        const int d = t * DPT + k;
        gtot[k] = d < D ? total[d] : 0;
        goff[k] = d < D ? off[(size_t)d * nblocks + blockIdx.x] : 0;
    }
    for (int w = 0; w < RS_WAVES; ++w)
        for (int d = t; d < D; d += RS_THREADS) s_wc[w][d] = 0;
    __syncthreads();
    // rank among the wavefront's keys of the same digit: every lane reads the digit's
    // count, then the digit's first lane writes the new one, then the next round reads.
    // The fences order these accesses among the wavefront's lanes; a wavefront's LDS
    // operations are executed in order anyway, so they cost 2 % of a sort at most.
    {
        unsigned short* wc = s_wc[wv];
        const unsigned long long lt = (1ull << lane) - 1ull;
#pragma unroll
        for (int r = 0; r < RS_ROUNDS; ++r)
        {
            const bool valid = key[r] >= 0;
            const int dig = (key[r] >> shift) & (D - 1);
            unsigned long long peers = __ballot(valid);  // lanes that hold the same digit
#pragma unroll
            for (int b = 0; b < BITS; ++b)
            {
                const unsigned long long m = __ballot((dig >> b) & 1);
                peers &= ((dig >> b) & 1) ? m : ~m;
            }
            rank[r] = wc[dig] + __popcll(peers & lt);
            wave_sync();
            if (valid && (peers & lt) == 0) wc[dig] = (unsigned short)(rank[r] + __popcll(peers));
            wave_sync();
        }
    }
    __syncthreads();
    // per digit: the wavefronts' keys in order, and the digits in order, in the tile
    // (local) and in the output (global)
    int cnt[DPT], lsum = 0, gsum = 0;
#pragma unroll
    for (int k = 0; k < DPT; ++k)
    {
        const int d = t * DPT + k;
        cnt[k] = 0;
        if (d < D)
            for (int w = 0; w < RS_WAVES; ++w) cnt[k] += s_wc[w][d];
        lsum += cnt[k];
        gsum += gtot[k];
    }
    const int linc = wave_inclusive_sum(lsum, lane), ginc = wave_inclusive_sum(gsum, lane);
    if (lane == 63)
    {
        s_wl[wv] = linc;
        s_wt[wv] = ginc;
    }
    __syncthreads();
    int lrun = linc - lsum, grun = ginc - gsum;
#pragma unroll
    for (int w = 0; w < RS_WAVES; ++w)
    {
        lrun += w < wv ? s_wl[w] : 0;
        grun += w < wv ? s_wt[w] : 0;
    }
#pragma unroll
    for (int k = 0; k < DPT; ++k)
    {
        const int d = t * DPT + k;
        if (d < D)
        {
            s_gofs[d] = grun + goff[k] - lrun;
            int at = lrun;
            for (int w = 0; w < RS_WAVES; ++w)
            {
                const int c = s_wc[w][d];
                s_wc[w][d] = (unsigned short)at;
                at += c;
            }
        }
        lrun += cnt[k];
        grun += gtot[k];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r)
        if (key[r] >= 0)
        {
            const int at = s_wc[wv][(key[r] >> shift) & (D - 1)] + rank[r];
            s_key[at] = key[r];
            s_val[at] = val[r];
        }
    __syncthreads();
    const int m = min(RS_TILE, n - i0);
#pragma unroll
    for (int r = 0; r < RS_ROUNDS; ++r)
    {
        const int at = r * RS_THREADS + t;
        if (at < m)
        {
            const int k = s_key[at];
            const int pos = s_gofs[(k >> shift) & (D - 1)] + at;
            keys_out[pos] = k;
            vals_out[pos] = s_val[at];
        }
    }
}

template <int BITS>
void radix_pass(const ibamr_plan* P, const int* kin, const int* vin, int n, int shift, int* ko, int* vo, hipStream_t s)
{
    const int nblk = (n + RS_TILE - 1) / RS_TILE;
    hipLaunchKernelGGL(k_rs_hist<BITS>, dim3(nblk), dim3(RS_THREADS), 0, s, kin, n, shift, nblk, P->rs_hist_d);
    hipLaunchKernelGGL(k_rs_scan, dim3(1 << BITS), dim3(256), 0, s, P->rs_hist_d, nblk, P->rs_off_d, P->rs_total_d);
    hipLaunchKernelGGL(k_rs_scatter<BITS>, dim3(nblk), dim3(RS_THREADS), 0, s, kin, vin, n, shift, nblk, P->rs_off_d,
                       P->rs_total_d, ko, vo);
}

// start[b] = first sorted position whose key is >= b, for b in [0, m] (keys in
// [0, m)): one binary search per bin, so the work per thread stays bounded
// however the points are spread over the bins.  nactive (if not null) counts the
// superbins (8 bins, before the sentinel m - 1) that hold points: one atomic per
// workgroup that has any, into a counter that k_bin_keys cleared.
__global__ void k_bin_bounds(const int* __restrict__ keys_sorted, int n, int m, int ksub, int* __restrict__ start,
                             int* __restrict__ nactive)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    int lo = 0, hi = b <= m ? n : 0;
    while (lo < hi)
    {
        const int mid = (lo + hi) >> 1;
        if ((keys_sorted[mid] >> ksub) < b)
            lo = mid + 1;
        else
            hi = mid;
    }
    if (b <= m) start[b] = lo;
    if (!nactive) return;
    // the first point at or after the superbin's first bin lies in one of its bins
    const bool some = (b & 7) == 0 && b < m - 1 && lo < n && (keys_sorted[lo] >> ksub) < b + 8;
    const int count = __syncthreads_count(some);
    if (threadIdx.x == 0 && count > 0) atomicAdd(nactive, count);
}

// out[ndim * p + d] = coordinate d of point p's cell (caller's order)
__global__ void k_cells_out(const int4* __restrict__ cell, int n, int ndim, int* __restrict__ out)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const int4 c = cell[p];
    out[(size_t)ndim * p] = c.x;
    out[(size_t)ndim * p + 1] = c.y;
    if (ndim == 3) out[(size_t)ndim * p + 2] = c.z;
}

// cells in bin order, and the inverse permutation (slot of every point)
__global__ void k_gather_cells(const int* __restrict__ perm, const int4* __restrict__ cell, int n,
                               int4* __restrict__ out, int* __restrict__ inv)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int p = perm[i];
    out[i] = cell[p];
    inv[p] = i;
}
} // namespace

// Stable LSD radix sort of n (key, value) pairs, keys in [0, 2^nbits).  vin ==
// nullptr: value i for element i.  The result lands in (kout, vout); (kt, vt)
// is the ping-pong pair.  Inputs are read in the first pass only.
int radix_sort_pairs(const ibamr_plan* P, const int* kin, const int* vin, int n, int nbits, int* kout, int* vout,
                     int* kt, int* vt, hipStream_t s)
{
    // As few passes as digits of RS_MAX_BITS allow, of equal digits.
    const int passes = std::max(1, (nbits + RS_MAX_BITS - 1) / RS_MAX_BITS);
    const int bits = (nbits + passes - 1) / passes;
    static_assert(RS_MAX_BITS == 10, "a pass for every digit width");
    for (int p = 0; p < passes; ++p)
    {
        const bool last_parity = ((passes - 1 - p) & 1) == 0;
        int* ko = last_parity ? kout : kt;
        int* vo = last_parity ? vout : vt;
        if (bits <= 8)
            radix_pass<8>(P, kin, vin, n, p * 8, ko, vo, s);
        else if (bits == 9)
            radix_pass<9>(P, kin, vin, n, p * 9, ko, vo, s);
        else
            radix_pass<10>(P, kin, vin, n, p * 10, ko, vo, s);
        HIP_OK(hipGetLastError());
        kin = ko;
        vin = vo;
    }
    return IBAMR_OK;
}

int bits_for(int maxkey)
{
    int nbits = 1;
    while (nbits < 31 && (maxkey >> nbits) != 0) ++nbits;
    return nbits;
}
} // namespace ibamr

extern "C" {

int ibamr_plan_bin_async(ibamr_plan* P, const double* X, int npoints, void* stream)
{
    if (!P) return fail(IBAMR_ERR_INVALID, "null plan");
    if (npoints < 0) return fail(IBAMR_ERR_INVALID, "npoints < 0");
    if (npoints > P->max_points) return fail(IBAMR_ERR_CAPACITY, "more points than the plan capacity");
    if (npoints > 0 && !X) return fail(IBAMR_ERR_INVALID, "null X");
    hipStream_t s = static_cast<hipStream_t>(stream);
    P->npoints = npoints;
    P->xs_valid = false;
    P->ws_valid = false;
    const int B = 256;
    const int m = P->nmem + 1;  // bins plus the out-of-domain sentinel
    if (npoints == 0)
    {
        hipLaunchKernelGGL(k_fill_int, dim3((m + 1 + B - 1) / B), dim3(B), 0, s, P->bin_start_d, m + 1, 0);
        HIP_OK(hipGetLastError());
        return IBAMR_OK;
    }
    BinArgs a{};
    a.X = X;
    a.n = npoints;
    for (int d = 0; d < 3; ++d)
    {
        a.xlo[d] = P->dom_xlo[d];
        a.xhi[d] = P->dom_xhi[d];
        a.ref_lo[d] = P->ref_lo[d];
        a.ref_hi[d] = P->ref_hi[d];
        a.sel_lo[d] = P->sel_lo[d];
        a.sel_hi[d] = P->sel_hi[d];
        a.dx[d] = P->dx[d];
        a.dom_lo[d] = P->dom_lo[d];
        a.dom_hi[d] = P->dom_hi[d];
        a.nb[d] = P->nb[d];
        a.nsb[d] = P->nsb[d];
    }
    a.bin = P->bin;
    a.nmem = P->nmem;
    a.ksub = P->ksub;
    a.nactive = P->nactive_d;
    a.keys = P->keys_d;
    a.cell = P->cell_d;
    const int G = (npoints + B - 1) / B;
    if (P->ndim == 3)
        hipLaunchKernelGGL(k_bin_keys<3>, dim3(G), dim3(B), 0, s, a);
    else
        hipLaunchKernelGGL(k_bin_keys<2>, dim3(G), dim3(B), 0, s, a);
    HIP_OK(hipGetLastError());
    // stable radix sort of keys [0, nmem << ksub] over the bits they use, into (keys_sorted_d, perm_d)
    {
        const int rc = radix_sort_pairs(P, P->keys_d, nullptr, npoints, bits_for(P->nmem << P->ksub), P->keys_sorted_d,
                                        P->perm_d, P->keys2_d, P->idx_d, s);
        if (rc != IBAMR_OK) return rc;
    }
    hipLaunchKernelGGL(k_bin_bounds, dim3((m + 1 + B - 1) / B), dim3(B), 0, s, P->keys_sorted_d, npoints, m,
                       P->ksub, P->bin_start_d, P->nactive_d);
    HIP_OK(hipGetLastError());
    // idx_d is free once the sort is done: it now holds the inverse permutation
    hipLaunchKernelGGL(k_gather_cells, dim3(G), dim3(B), 0, s, P->perm_d, P->cell_d, npoints, P->cell_sorted_d,
                       P->idx_d);
    HIP_OK(hipGetLastError());
    return IBAMR_OK;
}

int ibamr_plan_check(ibamr_plan* P, void* stream)
{
    if (!P) return fail(IBAMR_ERR_INVALID, "null plan");
    if (P->npoints < 0) return fail(IBAMR_ERR_NOT_BINNED, "points not binned");
    hipStream_t s = static_cast<hipStream_t>(stream);
    int first_sentinel = 0;
    HIP_OK(hipMemcpyAsync(&first_sentinel, P->bin_start_d + P->nmem, sizeof(int), hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    if (first_sentinel != P->npoints)
        return fail(IBAMR_ERR_OUT_OF_DOMAIN, std::to_string(P->npoints - first_sentinel) +
                                                 " point(s) outside the level domain (or NaN positions)");
    return IBAMR_OK;
}

int ibamr_plan_get_cell_indices(const ibamr_plan* P, int* cells, void* stream)
{
    if (!P || !cells) return fail(IBAMR_ERR_INVALID, "null argument");
    if (P->npoints < 0) return fail(IBAMR_ERR_NOT_BINNED, "points not binned");
    if (P->npoints == 0) return IBAMR_OK;
    const int B = 256;
    hipLaunchKernelGGL(k_cells_out, dim3((P->npoints + B - 1) / B), dim3(B), 0, static_cast<hipStream_t>(stream),
                       P->cell_d, P->npoints, P->ndim, cells);
    HIP_OK(hipGetLastError());
    return IBAMR_OK;
}

int ibamr_plan_bin(ibamr_plan* P, const double* X, int npoints, void* stream)
{
    const int rc = ibamr_plan_bin_async(P, X, npoints, stream);
    if (rc != IBAMR_OK) return rc;
    return ibamr_plan_check(P, stream);
}

} // extern "C"
