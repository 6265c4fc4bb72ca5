// le_spread3d.h -- 3-D spread kernel for gfx950 (included by le_spread.hip,
// which defines SpreadArgs, PatchDev and TileDesc).
//
// FP32C spread (k_spread3): owner-computes, register-resident.  One wavefront owns a
// column tile of one array: TX x TY (x, y) grid lines (8 x 8 or 16 x 4), one
// per lane, times ZC consecutive z values held in registers.  Points that can reach the
// tile are staged 64 at a time: each lane takes one point's stencil (the starts and
// weights that the set-up pass computed once per point) and writes the x and y weights,
// aligned to the tile's lanes and zero-padded, plus the z weights to LDS.  The staged
// points are then applied grouped by their first z index: a ballot per z start
// yields the points with that start, so every register index is a compile-time
// constant (no dynamic VGPR indexing).  Per point and lane the work is two LDS
// reads, one product and W fused multiply-adds.  No atomics: each grid value
// lives in one lane's register and receives its contributions in a fixed
// order, so results are bitwise reproducible.  Each chunk's contributions go to FP32
// partial sums, which are folded into FP64 totals after the chunk (a chunk holds at
// most 64 points, so the FP32 sums stay short).
// FP64 (k_spread3b) and FP32C columns swept along z (k_spread3s): see there.
#pragma once

namespace
{
// staged weight rows: the tile's TX (x) or TY (y) lanes, padded to an odd
// stride (no bank conflicts between the rows of different points)
template <int N>
constexpr int s3_pad()
{
    return N + 1;
}
constexpr int S3_MAXCOMB = 64;

// f(integral_constant<int, LO>) ... f(integral_constant<int, HI - 1>): arrays indexed
// by these constants become registers before any loop is unrolled
template <int LO, int HI, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (LO < HI)
    {
        f(std::integral_constant<int, LO>{});
        static_for<LO + 1, HI>(f);
    }
}
#define IBAMR_INLINE __attribute__((always_inline))

// a wave-uniform double, in scalar registers
__device__ __forceinline__ double uniform_double(double v)
{
    const int lo = __builtin_amdgcn_readfirstlane(__double2loint(v)), hi = __builtin_amdgcn_readfirstlane(__double2hiint(v));
    return __hiloint2double(hi, lo);
}

template <int KER, int ZC, int TX>
__global__ __launch_bounds__(64) void k_spread3(SpreadArgs<float> a)
{
    using T = float;
    using KT = KernelTraits<KER>;
    constexpr int W = KT::W;
    // the set-up pass's stencils are staged, except for kernels whose stencil side
    // depends on the unshifted X (an image's differs)
    constexpr bool PRECOMP = !side_by_unshifted_x<KER>();
    constexpr int TY = 64 / TX;  // the 64 lanes: TX x TY grid lines
    constexpr int PX = s3_pad<TX>(), PY = s3_pad<TY>();
    static_assert(TX * TY == 64, "one lane per grid line");
    __shared__ T s_rx[64 * PX];
    __shared__ T s_ry[64 * PY];
    __shared__ T s_wz[64 * 8];
    __shared__ int s_lb[3][16];
    __shared__ int s_lo[3][16];
    __shared__ int s_ln[3];
    __shared__ int s_cs[S3_MAXCOMB];    // per combination: first sorted point
    __shared__ int s_cl[S3_MAXCOMB];    //                  number of points
    __shared__ int s_co[S3_MAXCOMB];    //                  image offset code
    __shared__ int s_cp[S3_MAXCOMB + 1];// prefix of lengths

    const int lane = threadIdx.x;
    const int x = lane % TX, y = lane / TX;
    const TileDesc td = a.tiles[blockIdx.x];
    if (td.patch < 0) return;  // padding of the XCD-ordered work list
    const PatchDev P = a.patches[td.patch];
    const int axis = a.side ? td.comp : -1;
    const int tsz[3] = {TX, TY, ZC};
    int alo[3], ahi[3], an[3], flo[3], fhi[3];
    double xl[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        alo[d] = P.ilo[d] - a.gcw[d];
        ahi[d] = P.ihi[d] + a.gcw[d] + (d == axis ? 1 : 0);
        an[d] = ahi[d] - alo[d] + 1;
        flo[d] = alo[d] + td.t[d] * tsz[d];
        fhi[d] = min(flo[d] + tsz[d] - 1, ahi[d]);
        if (a.mode == IBAMR_SPREAD_ACCUMULATE_INTERIOR)
        {
            flo[d] = max(flo[d], P.ilo[d]);
            fhi[d] = min(fhi[d], P.ihi[d] + (d == axis ? 1 : 0));
        }
        xl[d] = P.xlo[d] - (d == axis ? 0.5 * a.dx[d] : 0.0);  // LEInteractor.cpp:3689
    }
    if (flo[0] > fhi[0] || flo[1] > fhi[1] || flo[2] > fhi[2]) return;  // tile wholly in the ghost region
    T* __restrict__ arr = a.arrays[td.patch * a.narr + (a.side ? td.comp : 0)];
    const size_t plane = (size_t)an[0] * an[1];
    if (!a.side) arr += (size_t)td.comp * plane * an[2];
    const int fcomp = td.comp;
    const int gx = flo[0] + x, gy = flo[1] + y;
    const bool col_in = gx <= fhi[0] && gy <= fhi[1];
    const size_t col_off = (size_t)(gx - alo[0]) + (size_t)an[0] * (size_t)(gy - alo[1]);

    // cells whose points can reach the tile, inside the patch's Lagrangian ghost box
    int clo[3], chi[3];
    bool any = true;
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        clo[d] = max(flo[d] - a.reach, P.ilo[d] - a.idx_gcw);
        chi[d] = min(fhi[d] + a.reach, P.ihi[d] + a.idx_gcw);
        any = any && clo[d] <= chi[d];
    }
    // per-axis (bin, image offset) lists in increasing (bin, offset) order
    if (lane < 3)
    {
        const int d = lane;
        int n = 0;
        if (any)
        {
            const int N = a.pshift[d];
            const int omax = N > 0 ? 1 : 0;
            for (int o = -omax; o <= omax; ++o)
            {
                const int pl = max(clo[d] - o * N, a.dom_lo[d]);
                const int ph = min(chi[d] - o * N, a.dom_hi[d]);
                if (pl > ph) continue;
                const int bl = floor_div(pl - a.dom_lo[d], a.bin);
                const int bh = floor_div(ph - a.dom_lo[d], a.bin);
                for (int b = bl; b <= bh && n < 16; ++b)
                {
                    int k = n++;
                    while (k > 0 && (s_lb[d][k - 1] > b || (s_lb[d][k - 1] == b && s_lo[d][k - 1] > o)))
                    {
                        s_lb[d][k] = s_lb[d][k - 1];
                        s_lo[d][k] = s_lo[d][k - 1];
                        --k;
                    }
                    s_lb[d][k] = b;
                    s_lo[d][k] = o;
                }
            }
        }
        s_ln[d] = n;
    }
    __syncthreads();
    const int nx = s_ln[0], ny = s_ln[1], nz = s_ln[2];
    const int ncomb = nx * ny * nz;

    // registers: tile values, accumulated in FP64, plus the chunk's FP32 partial sums
    double acc[ZC];
    T part[ZC];
    const bool overwrite = a.mode == IBAMR_SPREAD_OVERWRITE;
#pragma unroll
    for (int z = 0; z < ZC; ++z)
    {
        acc[z] = 0.0;
        part[z] = T(0);
    }

    // total number of points in the visited bins; an empty tile keeps its values.
    // The lane's combination of the first group is kept for the chunk loop.
    int total = 0, g0_st = 0, g0_ln = 0, g0_oc = 0;
    for (int c = lane; c < ncomb; c += 64)
    {
        const int kx = c % nx, ky = (c / nx) % ny, kz = c / (nx * ny);
        const int m = bin_mem(3, s_lb[0][kx], s_lb[1][ky], s_lb[2][kz], a.nb, a.nsb);
        const int st = a.bin_start[m], ln = a.bin_start[m + 1] - st;
        total += ln;
        if (c == lane)
        {
            g0_st = st;
            g0_ln = ln;
            g0_oc = (s_lo[0][kx] + 1) + 3 * (s_lo[1][ky] + 1) + 9 * (s_lo[2][kz] + 1);
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) total += __shfl_xor(total, off);
    if (total == 0 && !overwrite) return;
    // LDataManager::spread (interior mode) spreads into zeroed data and adds the
    // old values afterwards (LDataManager.cpp:594, 661-663); the raw
    // LEInteractor::spread (accumulate mode) adds each contribution to the
    // existing value (f.m4:1463)
    const bool from_old = a.mode == IBAMR_SPREAD_ACCUMULATE;
    if (from_old && col_in)
    {
#pragma unroll
        for (int z = 0; z < ZC; ++z)
            if (flo[2] + z <= fhi[2]) acc[z] = (double)arr[col_off + plane * (size_t)(flo[2] + z - alo[2])];
    }

    const T inv_vol = T(1.0 / a.vol);
    for (int cb = 0; cb < ncomb && total > 0; cb += S3_MAXCOMB)
    {
        // ---- this group of combinations: ranges and their prefix (in canonical order)
        {
            const int c = cb + lane;
            int st = cb == 0 ? g0_st : 0, ln = cb == 0 ? g0_ln : 0, oc = cb == 0 ? g0_oc : 0;
            if (cb > 0 && lane < S3_MAXCOMB && c < ncomb)
            {
                const int kx = c % nx, ky = (c / nx) % ny, kz = c / (nx * ny);
                const int m = bin_mem(3, s_lb[0][kx], s_lb[1][ky], s_lb[2][kz], a.nb, a.nsb);
                st = a.bin_start[m];
                ln = a.bin_start[m + 1] - st;
                oc = (s_lo[0][kx] + 1) + 3 * (s_lo[1][ky] + 1) + 9 * (s_lo[2][kz] + 1);
            }
            // inclusive scan of ln across the wavefront
            int inc = ln;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1)
            {
                const int t = __shfl_up(inc, off);
                if (lane >= off) inc += t;
            }
            if (lane < S3_MAXCOMB)
            {
                s_cs[lane] = st;
                s_cl[lane] = ln;
                s_co[lane] = oc;
                s_cp[lane + 1] = inc;
            }
            if (lane == 0) s_cp[0] = 0;
        }
        __syncthreads();
        const int ngc = min(S3_MAXCOMB, ncomb - cb);
        const int gtotal = s_cp[ngc];

        // chunks: any 64 consecutive points of the group.  The next chunk's point
        // data is loaded while the current one is applied.
        int cq = 0;
        auto lane_point = [&](int& k, int& oc) {
            k = -1;
            oc = 13;
            const int q = cq + lane;
            if (q < gtotal)
            {
                int lo = 0, hi = ngc - 1;  // last combination with prefix <= q
                while (lo < hi)
                {
                    const int mid = (lo + hi + 1) >> 1;
                    if (s_cp[mid] <= q)
                        lo = mid;
                    else
                        hi = mid - 1;
                }
                k = s_cs[lo] + (q - s_cp[lo]);
                oc = s_co[lo];
            }
        };
        bool cvalid = cq < gtotal;
        int nk, noc;
        int4 nc4 = make_int4(0, 0, 0, 0);
        double nX[3] = {0.0, 0.0, 0.0};
        T nF = T(0);
        int nst[3] = {0, 0, 0};   // precomputed stencil starts and weights
        float nw[3][W];
        // the lane's point of the current chunk: precomputed starts and weights (rows
        // of the point's axis variants) or position, F, cell
        auto load_point = [&]() {
            if (nk < 0) return;
            nc4 = a.cells[nk];
            if (!PRECOMP)
            {
#pragma unroll
                for (int d = 0; d < 3; ++d) nX[d] = a.X[3 * (size_t)nk + d];
            }
            else
            {
#pragma unroll
                for (int d = 0; d < 3; ++d)
                {
                    const int v = (a.nvar == 2 && d == axis) ? 1 : 0;
                    const size_t row = (size_t)(d * a.nvar + v) * a.npts + nk;
                    nst[d] = a.st[row];
#pragma unroll
                    for (int j = 0; j < W; ++j) nw[d][j] = a.wt[row * W + j];
                }
            }
            nF = a.F[(size_t)a.fdepth * nk + fcomp];
        };
        lane_point(nk, noc);
        load_point();
        while (cvalid)
        {
            const int k = nk, oc = noc;
            const int4 c4 = nc4;
            const T Fv = nF;

            int my_zz = 1 << 20;
            if (k >= 0)
            {
                const int o[3] = {oc % 3 - 1, (oc / 3) % 3 - 1, oc / 9 - 1};
                const int cc[3] = {c4.x, c4.y, c4.z};
                bool ok = true;
#pragma unroll
                for (int d = 0; d < 3; ++d)
                {
                    const int ci = cc[d] + o[d] * a.pshift[d];
                    ok = ok && ci >= clo[d] && ci <= chi[d];
                }
                if (ok)
                {
                    T w[3][W];
                    int bse[3];
                    if (!PRECOMP)
                    {
#pragma unroll
                        for (int d = 0; d < 3; ++d)
                        {
                            // X + Xshift, Xshift = (double)(offset) * dx  (LIndexSetData.cpp:116)
                            const double Xs = nX[d] + (double)(o[d] * a.pshift[d]) * a.dx[d];
                            bse[d] = P.ilo[d] + weights_1d_u<KER>(Xs, nX[d], xl[d], a.dx[d], w[d]);
                        }
                    }
                    else
                    {
                        // precomputed in the level's frame (k_point_weights); an image
                        // moves the stencil by whole periods
#pragma unroll
                        for (int d = 0; d < 3; ++d)
                        {
                            bse[d] = nst[d] + o[d] * a.pshift[d];
#pragma unroll
                            for (int j = 0; j < W; ++j) w[d][j] = (T)nw[d][j];
                        }
                    }
                    const int dx0 = bse[0] - flo[0], dy0 = bse[1] - flo[1], zz = bse[2] - flo[2];
                    if (dx0 > -W && dx0 < TX && dy0 > -W && dy0 < TY && zz > -W && zz < ZC)
                    {
                        // rows hold the weight of each of the tile's 8 x (y) lanes, zero outside the stencil
                        T* rx = s_rx + lane * PX;
                        T* ry = s_ry + lane * PY;
#pragma unroll
                        for (int i = 0; i < TX; ++i) rx[i] = T(0);
#pragma unroll
                        for (int i = 0; i < TY; ++i) ry[i] = T(0);
                        const T fx = KT::IB ? Fv : Fv * inv_vol;
#pragma unroll
                        for (int j = 0; j < W; ++j)
                        {
                            if ((unsigned)(dx0 + j) < (unsigned)TX) rx[dx0 + j] = w[0][j] * fx;
                            if ((unsigned)(dy0 + j) < (unsigned)TY) ry[dy0 + j] = w[1][j];
                            s_wz[lane * 8 + j] = KT::IB ? w[2][j] * inv_vol : w[2][j];
                        }
                        my_zz = zz;
                    }
                }
            }
            __syncthreads();
            // advance, and load the next chunk's points while this one is applied
            cq += 64;
            cvalid = cq < gtotal;
            nk = -1;
            if (cvalid) lane_point(nk, noc);
            load_point();
            const bool chunk_any = __ballot(my_zz < (1 << 20)) != 0;
            if (chunk_any)
            {
#pragma unroll
                for (int zz = -(W - 1); zz < ZC; ++zz)
                {
                    unsigned long long m = __ballot(my_zz == zz);
                    while (m)
                    {
                        // two points per step so their LDS reads overlap
                        const int j = __builtin_ctzll(m);
                        m &= m - 1;
                        const int j2 = m ? __builtin_ctzll(m) : j;
                        const bool two = m != 0;
                        if (two) m &= m - 1;
                        const T wx = s_rx[j * PX + x];
                        const T wy = s_ry[j * PY + y];
                        const T wx2 = s_rx[j2 * PX + x];
                        const T wy2 = s_ry[j2 * PY + y];
                        T wz[W], wz2[W];
#pragma unroll
                        for (int i = 0; i < W; ++i)
                        {
                            wz[i] = s_wz[j * 8 + i];
                            wz2[i] = s_wz[j2 * 8 + i];
                        }
                        const T b = wx * wy;
                        const T b2 = two ? wx2 * wy2 : T(0);
#pragma unroll
                        for (int i = 0; i < W; ++i)
                            if (zz + i >= 0 && zz + i < ZC)
                                part[zz + i] = fmaf(b2, wz2[i], fmaf(b, wz[i], part[zz + i]));
                    }
                }
                // fold the chunk's partial sums into the FP64 totals
#pragma unroll
                for (int z = 0; z < ZC; ++z)
                {
                    acc[z] = acc[z] + (double)part[z];
                    part[z] = T(0);
                }
            }
            __syncthreads();
        }
    }

    if (col_in)
    {
#pragma unroll
        for (int z = 0; z < ZC; ++z)
            if (flo[2] + z <= fhi[2])
            {
                T* v = arr + col_off + plane * (size_t)(flo[2] + z - alo[2]);
                *v = (overwrite || from_old) ? (T)acc[z] : (T)((double)*v + acc[z]);
            }
    }
}


// ----------------------------------------------------------------------------- FP64: batches of hits

// FP64 spread (k_spread3b): owner-computes, register-resident.  One wavefront owns
// a tile of one array: 8 x 8 (or 16 x 4) grid lines, one per lane, times ZC values
// along z in registers.  Points are taken in three steps, so that each step runs
// on full wavefronts although few candidates of a bin reach a tile (uniform points
// of a 512^3 level: 16 points a bin, 5 of them in reach):
//   filter  64 candidates of the reachable bins at a time (chunks cross bins):
//           cell inside the reachable box, position near enough; the others go
//           into a ring in LDS, in bin order;
//   stage   up to 64 ring entries, one per lane, whole chunks of a bin: the
//           reference's weights (quotients by dx and vol from reciprocals, div_by),
//           each entry's place in the order of summation, its record to LDS there;
//   apply   the records one after another: per lane two weights, the W z weights
//           and F from LDS, the reference's products, W additions into registers.
//           The loop runs over the z starts, so register indices are constants.
// Order per value (fixed by the bins, whatever the tile): bin and image, 64-point
// chunk of the bin, z start, rank.
// Bound by VALU issue and LDS returns: per point and tile 48 VALU instructions
// (24 of them FP64 products and sums for IB_6; 36 of the 64 lanes at most lie under
// a stencil) and 36 cycles of the CU's LDS path.  512^3 IB_6, 8.4 M points: 9.4 ms
// (67 % of the VALU cycles); 16.5 ms when each 64-point chunk of a bin was staged
// by itself, weights evaluated for a few lanes.  Not faster: four waves per SIMD
// instead of three (LDS), a switch over the z starts (accumulators in scratch).
template <int KER, int ZC, int TX>
__global__ __launch_bounds__(64, ZC <= 16 ? 4 : 3) void k_spread3b(SpreadArgs<double> a)
{
    using KT = KernelTraits<KER>;
    constexpr int W = KT::W;
    constexpr int TY = 64 / TX;
    constexpr int NREC = 3 * W + 1;                  // x, y, z weights and F of a hit
    constexpr int ROW = NREC % 2 ? NREC : NREC + 1;  // odd: rows written by 64 lanes without bank conflicts
    constexpr int QCAP = 128;
    static_assert(TX * TY == 64 && ZC + W - 1 <= 64, "one lane per grid line; 6-bit keys");
    __shared__ double s_row[64 * ROW];
    __shared__ int s_info[64];
    __shared__ int s_qk[QCAP], s_qg[QCAP];  // ring of candidates in reach: point, (combination, chunk of its bin)
    __shared__ unsigned char s_qo[QCAP];    //                              image code
    __shared__ int s_lb[3][16];
    __shared__ int s_lo[3][16];
    __shared__ int s_ln[3];
    __shared__ int s_cs[64];                // per combination of the group: first point - first position
    __shared__ int s_cf[64];                //                               first position
    __shared__ int s_co[64];                //                               image code

    const int lane = threadIdx.x;
    const int x = lane % TX, y = lane / TX;
    const TileDesc td = a.tiles[blockIdx.x];
    if (td.patch < 0) return;  // padding of the XCD-ordered work list
    const PatchDev P = a.patches[td.patch];
    const int axis = a.side ? td.comp : -1;
    const int tsz[3] = {TX, TY, ZC};
    int alo[3], ahi[3], an[3], flo[3], fhi[3];
    double xl[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        alo[d] = P.ilo[d] - a.gcw[d];
        ahi[d] = P.ihi[d] + a.gcw[d] + (d == axis ? 1 : 0);
        an[d] = ahi[d] - alo[d] + 1;
        flo[d] = alo[d] + td.t[d] * tsz[d];
        fhi[d] = min(flo[d] + tsz[d] - 1, ahi[d]);
        if (a.mode == IBAMR_SPREAD_ACCUMULATE_INTERIOR)
        {
            flo[d] = max(flo[d], P.ilo[d]);
            fhi[d] = min(fhi[d], P.ihi[d] + (d == axis ? 1 : 0));
        }
        xl[d] = P.xlo[d] - (d == axis ? 0.5 * a.dx[d] : 0.0);  // LEInteractor.cpp:3689
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) xl[d] = uniform_double(xl[d]);
    if (flo[0] > fhi[0] || flo[1] > fhi[1] || flo[2] > fhi[2]) return;  // tile wholly in the ghost region
    double* __restrict__ arr = a.arrays[td.patch * a.narr + (a.side ? td.comp : 0)];
    const size_t plane = (size_t)an[0] * an[1];
    if (!a.side) arr += (size_t)td.comp * plane * an[2];
    const int fcomp = td.comp;
    const int gx = flo[0] + x, gy = flo[1] + y;
    const bool col_in = gx <= fhi[0] && gy <= fhi[1];
    const size_t col_off = (size_t)(gx - alo[0]) + (size_t)an[0] * (size_t)(gy - alo[1]);

    // cells whose points can reach the tile, inside the patch's Lagrangian ghost box
    int clo[3], chi[3];
    bool any = true;
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        clo[d] = max(flo[d] - a.reach, P.ilo[d] - a.idx_gcw);
        chi[d] = min(fhi[d] + a.reach, P.ihi[d] + a.idx_gcw);
        any = any && clo[d] <= chi[d];
    }
    // per-axis (bin, image offset) lists in increasing (bin, offset) order
    if (lane < 3)
    {
        const int d = lane;
        int n = 0;
        if (any)
        {
            const int N = a.pshift[d];
            const int omax = N > 0 ? 1 : 0;
            for (int o = -omax; o <= omax; ++o)
            {
                const int pl = max(clo[d] - o * N, a.dom_lo[d]);
                const int ph = min(chi[d] - o * N, a.dom_hi[d]);
                if (pl > ph) continue;
                const int bl = floor_div(pl - a.dom_lo[d], a.bin);
                const int bh = floor_div(ph - a.dom_lo[d], a.bin);
                for (int b = bl; b <= bh && n < 16; ++b)
                {
                    int k = n++;
                    while (k > 0 && (s_lb[d][k - 1] > b || (s_lb[d][k - 1] == b && s_lo[d][k - 1] > o)))
                    {
                        s_lb[d][k] = s_lb[d][k - 1];
                        s_lo[d][k] = s_lo[d][k - 1];
                        --k;
                    }
                    s_lb[d][k] = b;
                    s_lo[d][k] = o;
                }
            }
        }
        s_ln[d] = n;
    }
    __syncthreads();
    const int nx = __builtin_amdgcn_readfirstlane(s_ln[0]), ny = __builtin_amdgcn_readfirstlane(s_ln[1]),
              nz = __builtin_amdgcn_readfirstlane(s_ln[2]);
    const int ncomb = nx * ny * nz;

    // the lane's combination c of the canonical (z, y, x) order: its points and image code
    auto combination = [&](int c, int& st, int& ln, int& oc) {
        st = ln = oc = 0;
        if (c >= ncomb) return;
        const int kx = c % nx, ky = (c / nx) % ny, kz = c / (nx * ny);
        const int m = bin_mem(3, s_lb[0][kx], s_lb[1][ky], s_lb[2][kz], a.nb, a.nsb);
        st = a.bin_start[m];
        ln = a.bin_start[m + 1] - st;
        oc = (s_lo[0][kx] + 1) + 3 * (s_lo[1][ky] + 1) + 9 * (s_lo[2][kz] + 1);
    };
    int g_st, g_ln, g_oc;
    combination(lane, g_st, g_ln, g_oc);
    int total = g_ln;
    for (int c = lane + 64; c < ncomb; c += 64)
    {
        int st, ln, oc;
        combination(c, st, ln, oc);
        total += ln;
    }
    const bool overwrite = a.mode == IBAMR_SPREAD_OVERWRITE;
    if (__ballot(total > 0) == 0 && !overwrite) return;  // an empty tile keeps its values

    double acc[ZC];
    // LDataManager::spread (interior mode) spreads into zeroed data and adds the
    // old values afterwards (LDataManager.cpp:594, 661-663); the raw
    // LEInteractor::spread (accumulate mode) adds each contribution to the
    // existing value (f.m4:1463)
    const bool from_old = a.mode == IBAMR_SPREAD_ACCUMULATE;
    static_for<0, ZC>([&](auto zc) IBAMR_INLINE {
        constexpr int z = decltype(zc)::value;
        acc[z] = 0.0;
        if (from_old && col_in && flo[2] + z <= fhi[2]) acc[z] = arr[col_off + plane * (size_t)(flo[2] + z - alo[2])];
    });

    const double vol = a.vol, rvol = a.rvol;
    int xp = x + 8, yp = y + 8;
    asm("" : "+v"(xp), "+v"(yp));  // one subtraction each per hit
    const unsigned long long lt = (1ull << lane) - 1ull;

    // ---- the stream of candidates: the combinations in canonical order, 64 of them
    // (a group) at a time
    int cb = -64, cq = 0, gtotal = 0, lex = 0;  // group, position in it, its points, the lane's first position
    int cf = 0;                                 // the combination holding the next position to fetch
    int nk = -1, noc = 13, ng = 0;
    int4 nc4 = make_int4(0, 0, 0, 0);
    double nX[3] = {0.0, 0.0, 0.0};
    auto fetch = [&](int q0) __attribute__((always_inline)) {
        const int q = q0 + lane, ngc = min(64, ncomb - cb);
        int comb = cf, ncf = cf;
        for (int c = cf + 1; c < ngc; ++c)
        {
            const int e = __builtin_amdgcn_readlane(lex, c);
            if (e > q0 + 64) break;
            ncf = c;
            comb += e <= q ? 1 : 0;
        }
        cf = ncf;  // holds position q0 + 64, the next batch's first
        nk = -1;
        if (q >= gtotal) return;
        nk = q + s_cs[comb];
        noc = s_co[comb];
        ng = (cb >> 6) << 25 | comb << 19 | (((q - s_cf[comb]) >> 6) & 0x7ffff);
        nc4 = a.cells[nk];
#pragma unroll
        for (int d = 0; d < 3; ++d) nX[d] = a.X[3 * (size_t)nk + d];
    };
    // the range of (X - x_lower) / dx - (flo - ilo) whose stencils reach the tile,
    // widened by what FP32 rounds (the exact test follows with the weights)
    float thi[3];
    const float tlo = (float)reach_lo<KER>() - 1e-3f;
#pragma unroll
    for (int d = 0; d < 3; ++d) thi[d] = (float)(fhi[d] - flo[d]) + (float)reach_hi<KER>() + 1e-3f;
    bool more = true, live = true;
    int qh = 0, qn = 0;         // the ring's first entry and length
    int nh = 0, infos = 0xff;   // the batch being applied: its hits; hit j's place and z start in lane j
    int j = 0, info = 0xff;     // the next hit
    do
    {
        if (j >= nh)
        {
            // ---- fill the ring
            while (more && qn < 64)
            {
                if (cq >= gtotal)
                {
                    cb += 64;
                    if (cb >= ncomb)
                    {
                        more = false;
                        break;
                    }
                    if (cb > 0) combination(cb + lane, g_st, g_ln, g_oc);
                    int inc = g_ln;
#pragma unroll
                    for (int off = 1; off < 64; off <<= 1)
                    {
                        const int t = __shfl_up(inc, off);
                        if (lane >= off) inc += t;
                    }
                    lex = inc - g_ln;
                    gtotal = __builtin_amdgcn_readlane(inc, 63);
                    cq = cf = 0;
                    s_cs[lane] = g_st - lex;
                    s_cf[lane] = lex;
                    s_co[lane] = g_oc;
                    __syncthreads();
                    if (gtotal == 0) continue;
                    fetch(0);
                }
                // the fetched candidates; the next ones' data are loaded meanwhile
                const int k = nk, oc = noc, gd = ng;
                const int cc[3] = {nc4.x, nc4.y, nc4.z};
                const int o[3] = {oc % 3 - 1, (oc / 3) % 3 - 1, oc / 9 - 1};
                bool ok = k >= 0;
#pragma unroll
                for (int d = 0; d < 3; ++d)
                {
                    const int ci = cc[d] + o[d] * a.pshift[d];
                    ok = ok && ci >= clo[d] && ci <= chi[d];
                    const float t =
                        (float)((nX[d] - xl[d]) * a.rdx[d] + (double)(o[d] * a.pshift[d] + P.ilo[d] - flo[d]));
                    ok = ok && !(t < tlo) && !(t > thi[d]);  // (true for NaN)
                }
                cq += 64;
                if (cq < gtotal) fetch(cq);
                const unsigned long long m = __ballot(ok);
                if (ok)
                {
                    const int p = (qh + qn + __popcll(m & lt)) & (QCAP - 1);
                    s_qk[p] = k;
                    s_qg[p] = gd;
                    s_qo[p] = (unsigned char)oc;
                }
                qn += __popcll(m);
            }
            __syncthreads();
            // whole chunks only (a chunk's order of summation covers all its points):
            // up to the last chunk boundary within 64 entries.  Without one the first
            // 64 are one chunk, and that has no more than 64 points.
            int n = qn;
            if (qn >= 64)
            {
                const int q = qh + lane;
                const unsigned long long b =
                    __ballot(lane + 1 < qn && s_qg[(q + 1) & (QCAP - 1)] != s_qg[q & (QCAP - 1)]);
                n = b ? 64 - __builtin_clzll(b) : 64;
            }
            // ---- stage them, one per lane: weights, place in the order of summation
            int key = 0, pos = 0;
            bool hit = false;
            double X[3] = {0.0, 0.0, 0.0}, Fv = 0.0;
            int dx0 = 0, dy0 = 0, oc = 13;
            int gid = -1;
            // X + Xshift, Xshift = (double)(offset) * dx  (LIndexSetData.cpp:116)
            auto weights = [&](int d, double* w) IBAMR_INLINE {
                const int o = (d == 0 ? oc % 3 : d == 1 ? (oc / 3) % 3 : oc / 9) - 1;
                const double Xs = X[d] + (double)(o * a.pshift[d]) * a.dx[d];
                return weights_1d_q<KER>(Xs, X[d], xl[d], a.dx[d], w, DivideBy{a.dx_ok ? a.rdx[d] : 0.0});
            };
            if (lane < n)
            {
                const int q = (qh + lane) & (QCAP - 1);
                const int k = s_qk[q];
                oc = s_qo[q];
                gid = s_qg[q];
                int bse[3];
#pragma unroll
                for (int d = 0; d < 3; ++d)
                {
                    double w[W];
                    X[d] = a.X[3 * (size_t)k + d];
                    bse[d] = P.ilo[d] + weights(d, w);  // the start; the weights once the place is known
                }
                Fv = a.F[(size_t)a.fdepth * k + fcomp];
                dx0 = bse[0] - flo[0];
                dy0 = bse[1] - flo[1];
                const int zz = bse[2] - flo[2];
                hit = dx0 > -W && dx0 < TX && dy0 > -W && dy0 < TY && zz > -W && zz < ZC;
                key = zz + W - 1;
            }
            const unsigned long long hits = __ballot(hit);
            nh = __builtin_amdgcn_readfirstlane(__popcll(hits));
            // order of summation: chunk of a bin, z start, rank.  The lanes are in
            // (chunk, rank) order, so inside each chunk's run of lanes: the hits with
            // a smaller z start, then those with the same one and a lower lane,
            // counted bit by bit of the z start.
            {
                const int before = __shfl_up(gid, 1);
                const unsigned long long first = __ballot(lane == 0 || gid != before);
                const unsigned long long upto = first & (lt | (1ull << lane));
                const unsigned long long beyond = first & ~(lt | (1ull << lane));
                const int g0 = 63 - __builtin_clzll(upto);
                const unsigned long long run_lt = (1ull << g0) - 1ull;
                const unsigned long long run_end = beyond ? (beyond & (~beyond + 1ull)) - 1ull : ~0ull;
                unsigned long long eq = hits & run_end & ~run_lt;
                pos = __popcll(hits & run_lt);
#pragma unroll
                for (int b = 5; b >= 0; --b)
                {
                    if ((ZC + W - 2) >> b == 0) continue;
                    const unsigned long long one = __ballot((key >> b) & 1);
                    if ((key >> b) & 1)
                    {
                        pos += __popcll(eq & ~one);
                        eq &= one;
                    }
                    else
                        eq &= ~one;
                }
                pos += __popcll(eq & lt);
            }
            if (hit)
            {
                // axis by axis (registers); safe: div_by rounds the quotients by vol correctly
                const double fa = fabs(Fv);
                bool safe = a.vol_div != 0 && (KT::IB || Fv == 0.0 || (fa >= 1e-100 && fa <= 1e100));
                double* r = s_row + pos * ROW;
#pragma unroll
                for (int d = 0; d < 3; ++d)
                {
                    double w[W];
                    weights(d, w);
#pragma unroll
                    for (int i = 0; i < W; ++i)
                    {
                        if (!KT::IB || d == 2)
                            safe = safe && (w[i] == 0.0 || (fabs(w[i]) >= 1e-40 && fabs(w[i]) <= 1e40));
                    }
#pragma unroll
                    for (int i = 0; i < W; ++i)
                    {
                        // IB folds 1/vol into w2 exactly as the reference (f.m4:1435)
                        if (KT::IB && d == 2) w[i] = safe ? div_by(w[i], vol, rvol) : w[i] / vol;
                        r[d * W + i] = w[i];
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                r[3 * W] = Fv;
                s_info[pos] = key | (dx0 + 8) << 8 | (dy0 + 8) << 16 | (safe ? 0 : 1 << 24);
            }
            __syncthreads();
            qh = (qh + n) & (QCAP - 1);
            qn -= n;
            infos = lane < nh ? s_info[lane] : 0xff;  // past the last hit: matches no z start
            j = 0;
            info = __builtin_amdgcn_readlane(infos, 0);
            live = n > 0;
        }
        // ---- a pass over the z starts takes the hits up to the next smaller one (a
        // chunk or two), so every register index is a compile-time constant
        static_for<-(W - 1), ZC>([&](auto zc) IBAMR_INLINE {
            constexpr int zz = decltype(zc)::value;
            while (__builtin_expect((info & 0xff) == zz + W - 1, 0))
            {
                const double* r = s_row + j * ROW;
                const int ix = xp - ((info >> 8) & 0xff), iy = yp - ((info >> 16) & 0xff);
                if ((unsigned)ix < (unsigned)W && (unsigned)iy < (unsigned)W)
                {
                    const double wx = r[ix], wy = r[W + iy], Fj = r[3 * W];
                    const double wxy = wx * wy;
                    const bool newton = !KT::IB && !(info >> 24);
                    // the W contributions side by side: each is a chain of dependent operations
                    double c[W];
                    static_for<0, W>([&](auto ic) IBAMR_INLINE {
                        constexpr int i = decltype(ic)::value;
                        c[i] = KT::IB ? wy * r[2 * W + i] : wxy * r[2 * W + i];
                    });
                    __builtin_amdgcn_sched_barrier(0);
                    if (KT::IB)
                    {
                        static_for<0, W>([&](auto ic) IBAMR_INLINE { c[decltype(ic)::value] = wx * c[decltype(ic)::value]; });
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    static_for<0, W>([&](auto ic) IBAMR_INLINE { c[decltype(ic)::value] = c[decltype(ic)::value] * Fj; });
                    __builtin_amdgcn_sched_barrier(0);
                    if (!KT::IB)  // over vol; one choice for the W quotients, which then run side by side
                    {
                        if (a.vol_div == 1)  // a power of two: the product rounds as the quotient does
                            static_for<0, W>([&](auto ic) IBAMR_INLINE { c[decltype(ic)::value] = c[decltype(ic)::value] * rvol; });
                        else if (newton)
                            static_for<0, W>([&](auto ic) IBAMR_INLINE { c[decltype(ic)::value] = div_by(c[decltype(ic)::value], vol, rvol); });
                        else
                            static_for<0, W>([&](auto ic) IBAMR_INLINE { c[decltype(ic)::value] = c[decltype(ic)::value] / vol; });
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    static_for<0, W>([&](auto ic) IBAMR_INLINE {
                        constexpr int i = decltype(ic)::value;
                        if constexpr (zz + i >= 0 && zz + i < ZC) acc[zz + i] = acc[zz + i] + c[i];
                    });
                }
                ++j;
                info = j < 64 ? __builtin_amdgcn_readlane(infos, j & 63) : 0xff;
            }
        });
    } while (live);
    if (col_in)
        static_for<0, ZC>([&](auto zc) IBAMR_INLINE {
            constexpr int z = decltype(zc)::value;
            if (flo[2] + z <= fhi[2])
            {
                double* v = arr + col_off + plane * (size_t)(flo[2] + z - alo[2]);
                *v = (overwrite || from_old) ? acc[z] : *v + acc[z];
            }
        });
}

// ----------------------------------------------------------------------------- FP32C: z sweep

// FP32C spread swept along z (k_spread3s): a wavefront owns TX x TY grid lines
// of one array over a long z segment and takes the z layers of bins (with
// their periodic images) in increasing z.  The segment's values pass through
// a window of S3S_ZW z values held in registers: before a layer is applied the
// window is placed at the layer's first reachable cell minus the stencil
// reach, so every stencil of the layer lies in the window whole (no z
// clipping; its first z value is one of S3S_ZW - W + 1 window positions), and
// the values below the new window position, which no later layer reaches, are
// written out.  A point is then applied once per xy tile instead of once per
// (xy tile, z tile), and staged once per column segment.  The layers' points
// form one stream of 64-point chunks (a chunk never spans two layers); the
// next chunk's point data and the next layer's bin ranges are loaded while the
// current chunk is applied.  Staging, ballots and the FP32 partials folded into
// FP64 totals are those of k_spread3; each value's summation order is fixed by
// the bins, the points' order and the tile shape.
constexpr int S3S_ZW = 16;    // z values in registers
constexpr int S3S_MAXZ = 64;  // z layers (bin, image) of one segment

template <int KER, int TX>
__global__ __launch_bounds__(64) void k_spread3s(SpreadArgs<float> a, int seg)
{
    using T = float;
    using KT = KernelTraits<KER>;
    constexpr int W = KT::W;
    constexpr int TY = 64 / TX;
    constexpr int PX = s3_pad<TX>(), PY = s3_pad<TY>();
    constexpr int ZW = S3S_ZW;
    constexpr int NZZ = ZW - W + 1;  // window positions of a stencil's first z value
    static_assert(TX * TY == 64, "one lane per grid line");
    // staged rows of the chunk's 64 points, plus row 64 of zeros (the partner
    // of the last point of a z start with an odd count)
    __shared__ T s_rx[65 * PX];
    __shared__ T s_ry[65 * PY];
    __shared__ __align__(16) T s_wz[65 * 8];
    __shared__ int s_lb[2][16];
    __shared__ int s_lo[2][16];
    __shared__ int s_ln[3];
    __shared__ int s_zb[S3S_MAXZ];  // z layers: bin, image offset; increasing shifted z
    __shared__ int s_zo[S3S_MAXZ];
    __shared__ int s_cd[64];        // per (x, y) combination of the layer: first sorted point - first position
    __shared__ int s_sx[64];        //                                      image shift in x (cells)
    __shared__ int s_sy[64];        //                                      image shift in y

    const int lane = threadIdx.x;
    const int x = lane % TX, y = lane / TX;
    const TileDesc td = a.tiles[blockIdx.x];
    if (td.patch < 0) return;  // padding of the XCD-ordered work list
    if (lane < PX) s_rx[64 * PX + lane] = T(0);
    if (lane < PY) s_ry[64 * PY + lane] = T(0);
    if (lane < 8) s_wz[64 * 8 + lane] = T(0);
    const PatchDev P = a.patches[td.patch];
    const int axis = a.side ? td.comp : -1;
    const int tsz[3] = {TX, TY, seg};
    int alo[3], ahi[3], an[3], flo[3], fhi[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        alo[d] = P.ilo[d] - a.gcw[d];
        ahi[d] = P.ihi[d] + a.gcw[d] + (d == axis ? 1 : 0);
        an[d] = ahi[d] - alo[d] + 1;
        flo[d] = alo[d] + td.t[d] * tsz[d];
        fhi[d] = min(flo[d] + tsz[d] - 1, ahi[d]);
        if (a.mode == IBAMR_SPREAD_ACCUMULATE_INTERIOR)
        {
            flo[d] = max(flo[d], P.ilo[d]);
            fhi[d] = min(fhi[d], P.ihi[d] + (d == axis ? 1 : 0));
        }
    }
    if (flo[0] > fhi[0] || flo[1] > fhi[1] || flo[2] > fhi[2]) return;  // tile wholly in the ghost region
    T* __restrict__ arr = a.arrays[td.patch * a.narr + (a.side ? td.comp : 0)];
    const size_t plane = (size_t)an[0] * an[1];
    if (!a.side) arr += (size_t)td.comp * plane * an[2];
    const int fcomp = td.comp;
    const int gx = flo[0] + x, gy = flo[1] + y;
    const bool col_in = gx <= fhi[0] && gy <= fhi[1];
    const size_t col_off = (size_t)(gx - alo[0]) + (size_t)an[0] * (size_t)(gy - alo[1]);

    // cells whose points can reach the tile, inside the patch's Lagrangian ghost box
    int clo[3], chi[3];
    bool any = true;
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        clo[d] = max(flo[d] - a.reach, P.ilo[d] - a.idx_gcw);
        chi[d] = min(fhi[d] + a.reach, P.ihi[d] + a.idx_gcw);
        any = any && clo[d] <= chi[d];
    }
    // x and y: (bin, image offset) lists in increasing (bin, offset) order; z:
    // layers with the offset outermost, so their shifted cells increase
    if (lane < 3)
    {
        const int d = lane;
        const int cap = d < 2 ? 16 : S3S_MAXZ;
        int n = 0;
        if (any)
        {
            const int N = a.pshift[d];
            const int omax = N > 0 ? 1 : 0;
            for (int o = -omax; o <= omax; ++o)
            {
                const int pl = max(clo[d] - o * N, a.dom_lo[d]);
                const int ph = min(chi[d] - o * N, a.dom_hi[d]);
                if (pl > ph) continue;
                const int bl = floor_div(pl - a.dom_lo[d], a.bin);
                const int bh = floor_div(ph - a.dom_lo[d], a.bin);
                for (int b = bl; b <= bh && n < cap; ++b)
                {
                    if (d == 2)
                    {
                        s_zb[n] = b;
                        s_zo[n] = o;
                        ++n;
                        continue;
                    }
                    int k = n++;
                    while (k > 0 && (s_lb[d][k - 1] > b || (s_lb[d][k - 1] == b && s_lo[d][k - 1] > o)))
                    {
                        s_lb[d][k] = s_lb[d][k - 1];
                        s_lo[d][k] = s_lo[d][k - 1];
                        --k;
                    }
                    s_lb[d][k] = b;
                    s_lo[d][k] = o;
                }
            }
        }
        s_ln[d] = n;
    }
    __syncthreads();
    const int nx = s_ln[0], ny = s_ln[1], nz = s_ln[2];
    const int nxy = nx * ny;  // at most 64 (the host admits only such shapes)

    double acc[ZW];
    T part[ZW];
#pragma unroll
    for (int z = 0; z < ZW; ++z)
    {
        acc[z] = 0.0;
        part[z] = T(0);
    }
    const bool overwrite = a.mode == IBAMR_SPREAD_OVERWRITE;
    // the raw LEInteractor::spread adds each contribution to the existing value
    // (f.m4:1463): the totals start from the old values; LDataManager::spread
    // (interior mode) spreads into zeroed data and adds the old values afterwards
    // (LDataManager.cpp:594, 661-663); overwrite replaces them
    const bool from_old = a.mode == IBAMR_SPREAD_ACCUMULATE;
    auto owned = [&](int z) { return col_in && z >= flo[2] && z <= fhi[2]; };
    auto at = [&](int z) { return arr + col_off + plane * (size_t)(z - alo[2]); };
    // the total a value starts from when it enters the window
    auto start = [&](int z) { return from_old && owned(z) ? (double)*at(z) : 0.0; };
    auto put = [&](int z, double v) {
        T* p = at(z);
        *p = (overwrite || from_old) ? (T)v : (T)((double)*p + v);
    };
    int wb = 0, zf = flo[2];  // window base; first value of the segment not yet written
    bool placed = false;
    // overwrite: values of the segment below z0 that were never in the window are zero
    auto zero_fill = [&](int z0) {
        if (overwrite && col_in)
            for (int z = zf; z < min(z0, fhi[2] + 1); ++z) *at(z) = T(0);
        zf = max(zf, z0);
    };
    auto load_window = [&]() {
#pragma unroll
        for (int i = 0; i < ZW; ++i) acc[i] = start(wb + i);
    };
    // moves the window base to nb (>= wb), writing the values that leave the window
    auto shift_to = [&](int nb) {
        if (!placed)
        {
            zero_fill(nb);
            wb = nb;
            placed = true;
            load_window();
            return;
        }
        const int sh = nb - wb;
        if (sh <= 0) return;
        if (sh >= ZW)
        {
#pragma unroll
            for (int i = 0; i < ZW; ++i)
                if (owned(wb + i) && wb + i >= zf) put(wb + i, acc[i]);
            zf = max(zf, wb + ZW);
            zero_fill(nb);
            wb = nb;
            load_window();
            return;
        }
        if (sh == 8)
        {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (owned(wb + i) && wb + i >= zf) put(wb + i, acc[i]);
#pragma unroll
            for (int i = 0; i < ZW; ++i) acc[i] = i + 8 < ZW ? acc[i + 8] : start(nb + i);
        }
        else
            for (int k = 0; k < sh; ++k)
            {
                if (owned(wb + k) && wb + k >= zf) put(wb + k, acc[0]);
#pragma unroll
                for (int i = 0; i < ZW - 1; ++i) acc[i] = acc[i + 1];
                acc[ZW - 1] = start(wb + k + ZW);
            }
        zf = max(zf, nb);
        wb = nb;
    };

    // ---- the chunk stream
    // bin_start values of the lane's (x, y) combination in layer ez (loads in flight until used)
    auto layer_range = [&](int ez, int& st, int& en) {
        st = 0;
        en = 0;
        if (ez < nz && lane < nxy)
        {
            const int m = bin_mem(3, s_lb[0][lane % nx], s_lb[1][lane / nx], s_zb[ez], a.nb, a.nsb);
            st = a.bin_start[m];
            en = a.bin_start[m + 1];
        }
    };
    int ez = -1, gtotal = 0;
    int lex = 0;   // lane c: first position of combination c in the layer's candidates
    int cf = 0;    // the combination holding the chunk's first position
    int pst, pen;  // the following layer's ranges
    layer_range(0, pst, pen);
    // moves to the next layer with points: its combinations' offsets into LDS
    auto next_layer = [&]() -> bool {
        while (++ez < nz)
        {
            const int st = pst, ln = pen - pst;
            layer_range(ez + 1, pst, pen);
            int inc = ln;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1)
            {
                const int t = __shfl_up(inc, off);
                if (lane >= off) inc += t;
            }
            lex = inc - ln;
            s_cd[lane] = st - lex;
            s_sx[lane] = lane < nxy ? s_lo[0][lane % nx] * a.pshift[0] : 0;
            s_sy[lane] = lane < nxy ? s_lo[1][lane / nx] * a.pshift[1] : 0;
            __syncthreads();
            gtotal = __builtin_amdgcn_readlane(inc, 63);
            cf = 0;
            if (gtotal > 0) return true;
        }
        return false;
    };
    // the lane's point of the chunk at cq: its index, image code, cell, stencil and F
    int cq = 0;
    int nk = -1, nsx = 0, nsy = 0;
    int4 nc4 = make_int4(0, 0, 0, 0);
    int nst[3] = {0, 0, 0};
    T nw[3][W];
    T nF = T(0);
    auto fetch = [&]() {
        // the lane's combination: cf plus the combinations after cf that start at
        // or before its position (offsets increase with the combination)
        const int q = cq + lane;
        int comb = cf, ncf = cf;
        for (int c = cf + 1; c < nxy; ++c)
        {
            const int e = __builtin_amdgcn_readlane(lex, c);
            if (e > cq + 64) break;
            ncf = c;
            comb += e <= q ? 1 : 0;
        }
        cf = ncf;  // holds position cq + 64, the next chunk's first
        nk = -1;
        if (q >= gtotal) return;
        nk = q + s_cd[comb];
        nsx = s_sx[comb];
        nsy = s_sy[comb];
        nc4 = a.cells[nk];
        // precomputed in the level's frame (k_point_weights)
#pragma unroll
        for (int d = 0; d < 3; ++d)
        {
            const int v = (a.nvar == 2 && d == axis) ? 1 : 0;
            const size_t row = (size_t)(d * a.nvar + v) * a.npts + nk;
            nst[d] = a.st[row];
#pragma unroll
            for (int j = 0; j < W; ++j) nw[d][j] = a.wt[row * W + j];
        }
        nF = a.F[(size_t)a.fdepth * nk + fcomp];
    };
    bool have = next_layer();
    if (have) fetch();
    const T iv = T(1.0 / a.vol);
    int zsh = 0;  // the layer's image shift in z (cells)
    while (have)
    {
        // a layer's first chunk: place the window for it
        if (cq == 0)
        {
            zsh = s_zo[ez] * a.pshift[2];
            shift_to(max(a.dom_lo[2] + s_zb[ez] * a.bin + zsh, clo[2]) - a.reach);
        }
        // ---- stage this chunk
        int my_zz = 1 << 20;
        if (nk >= 0)
        {
            const int sh[3] = {nsx, nsy, zsh};
            const int cc[3] = {nc4.x, nc4.y, nc4.z};
            bool ok = true;
            int bse[3];
#pragma unroll
            for (int d = 0; d < 3; ++d)
            {
                const int ci = cc[d] + sh[d];
                ok = ok && ci >= clo[d] && ci <= chi[d];
                bse[d] = nst[d] + sh[d];  // an image moves the stencil by whole periods
            }
            const int dx0 = bse[0] - flo[0], dy0 = bse[1] - flo[1], zz = bse[2] - wb;
            if (ok && dx0 > -W && dx0 < TX && dy0 > -W && dy0 < TY && zz >= 0 && zz < NZZ)
            {
                // rows hold the weight of each of the tile's x (y) lanes, zero outside the stencil
                T* rx = s_rx + lane * PX;
                T* ry = s_ry + lane * PY;
#pragma unroll
                for (int i = 0; i < TX; ++i) rx[i] = T(0);
#pragma unroll
                for (int i = 0; i < TY; ++i) ry[i] = T(0);
                const T fx = KT::IB ? nF : nF * iv;
                T wz[8];
#pragma unroll
                for (int j = 0; j < W; ++j)
                {
                    if ((unsigned)(dx0 + j) < (unsigned)TX) rx[dx0 + j] = nw[0][j] * fx;
                    if ((unsigned)(dy0 + j) < (unsigned)TY) ry[dy0 + j] = nw[1][j];
                    wz[j] = KT::IB ? nw[2][j] * iv : nw[2][j];
                }
#pragma unroll
                for (int j = W; j < 8; ++j) wz[j] = T(0);
                float4* wq = reinterpret_cast<float4*>(s_wz + lane * 8);
                wq[0] = make_float4(wz[0], wz[1], wz[2], wz[3]);
                if (W > 4) wq[1] = make_float4(wz[4], wz[5], wz[6], wz[7]);
                my_zz = zz;
            }
        }
        __syncthreads();
        // ---- the next chunk (its layer's ranges are already loaded): loads in flight
        cq += 64;
        if (cq >= gtotal)
        {
            cq = 0;
            have = next_layer();
        }
        if (have) fetch();
        // ---- apply this chunk
        if (__ballot(my_zz < (1 << 20)))
        {
#pragma unroll
            for (int zz = 0; zz < NZZ; ++zz)
            {
                unsigned long long m = __ballot(my_zz == zz);
                while (m)
                {
                    // two points per step so their LDS reads overlap
                    const int j = __builtin_ctzll(m);
                    m &= m - 1;
                    const int j2 = m ? __builtin_ctzll(m) : 64;
                    m &= m - 1;
                    const T wx = s_rx[j * PX + x];
                    const T wy = s_ry[j * PY + y];
                    const T wx2 = s_rx[j2 * PX + x];
                    const T wy2 = s_ry[j2 * PY + y];
                    T wz[W], wz2[W];
#pragma unroll
                    for (int i = 0; i < W; ++i)
                    {
                        wz[i] = s_wz[j * 8 + i];
                        wz2[i] = s_wz[j2 * 8 + i];
                    }
                    const T b = wx * wy;
                    const T b2 = wx2 * wy2;
#pragma unroll
                    for (int i = 0; i < W; ++i) part[zz + i] = fmaf(b2, wz2[i], fmaf(b, wz[i], part[zz + i]));
                }
            }
            // fold the chunk's partial sums into the FP64 totals
#pragma unroll
            for (int z = 0; z < ZW; ++z)
            {
                acc[z] = acc[z] + (double)part[z];
                part[z] = T(0);
            }
        }
        __syncthreads();
    }
    // the rest of the segment: the window's values, then zeros above it (overwrite)
    if (placed)
    {
#pragma unroll
        for (int i = 0; i < ZW; ++i)
            if (owned(wb + i) && wb + i >= zf) put(wb + i, acc[i]);
        zf = max(zf, wb + ZW);
    }
    zero_fill(fhi[2] + 1);
}

} // namespace
