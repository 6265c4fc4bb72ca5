// le_spread2d.h -- 2-D spread kernel for gfx950 (included by le_spread.hip after
// le_spread3d.h, whose SpreadArgs, static_for and uniform_double it uses).
//
// One wavefront owns an 8 x 8 tile of one array (NV = 1), one grid value per lane, or
// 16 x 16 (NV = 2, for few points on large levels), four values per lane 8 apart of
// which a stencil covers at most one, summed in FP64 in registers.  As in k_spread3b the
// points pass through three steps: 64 candidates of the reachable bins at a time are
// filtered by cell and position into a ring in LDS; up to 64 ring entries are staged, one per lane (weights, F); the
// staged points are then applied one after another, four at a time so that their
// LDS reads overlap: per lane two weights, two products and one addition.  Points
// come in the bins' order (bin y, image y, bin x, image x; rank), so every value's
// order of summation is fixed whatever the tile.
// Bound by the serial chain of a tile's points (latency; 2-D grids have few tiles), with
// few points on a large level by the number of workgroups.
#pragma once

namespace
{
constexpr int S2_TILE = 8;

template <int KER, typename T, int NV>
__global__ __launch_bounds__(64) void k_spread2(SpreadArgs<T> a)
{
    using KT = KernelTraits<KER>;
    constexpr int W = KT::W;
    constexpr int TILE = S2_TILE * NV;
    static_assert(W <= 8 && NV <= 2, "a stencil covers at most one of a lane's values along an axis");
    constexpr bool FP64 = sizeof(T) == 8;
    constexpr int NREC = 2 * W + 1;                  // x and y weights and F of a hit
    constexpr int ROW = NREC % 2 ? NREC : NREC + 1;  // odd: rows written by 64 lanes without bank conflicts
    constexpr int QCAP = 128, FAR = 64;              // FAR: a place no lane lies under
    __shared__ T s_row[64 * ROW];
    __shared__ int s_qk[QCAP];            // ring of candidates in reach: point,
    __shared__ unsigned char s_qo[QCAP];  //                              image code
    __shared__ int s_lb[2][16];
    __shared__ int s_lo[2][16];
    __shared__ int s_ln[2];
    __shared__ int s_cs[64];              // per combination of the group: first point - first position
    __shared__ int s_co[64];              //                               image code

    const int lane = threadIdx.x;
    const int x = lane & 7, y = lane >> 3;
    const TileDesc td = a.tiles[blockIdx.x];
    if (td.patch < 0) return;  // padding of the XCD-ordered work list
    const PatchDev P = a.patches[td.patch];
    const int axis = a.side ? td.comp : -1;
    int alo[2], ahi[2], an[2], flo[2], fhi[2];
    double xl[2];
#pragma unroll
    for (int d = 0; d < 2; ++d)
    {
        alo[d] = P.ilo[d] - a.gcw[d];
        ahi[d] = P.ihi[d] + a.gcw[d] + (d == axis ? 1 : 0);
        an[d] = ahi[d] - alo[d] + 1;
        flo[d] = alo[d] + td.t[d] * TILE;
        fhi[d] = min(flo[d] + TILE - 1, ahi[d]);
        if (a.mode == IBAMR_SPREAD_ACCUMULATE_INTERIOR)
        {
            flo[d] = max(flo[d], P.ilo[d]);
            fhi[d] = min(fhi[d], P.ihi[d] + (d == axis ? 1 : 0));
        }
        xl[d] = uniform_double(P.xlo[d] - (d == axis ? 0.5 * a.dx[d] : 0.0));  // LEInteractor.cpp:3689
    }
    if (flo[0] > fhi[0] || flo[1] > fhi[1]) return;  // tile wholly in the ghost region
    const int gx = flo[0] + x, gy = flo[1] + y;
    auto in = [&](int k) { return gx + 8 * (k % NV) <= fhi[0] && gy + 8 * (k / NV) <= fhi[1]; };  // value k of the lane
    T* __restrict__ arr = a.arrays[td.patch * a.narr + (a.side ? td.comp : 0)];
    if (!a.side) arr += (size_t)td.comp * an[0] * an[1];
    auto at = [&](int k) {
        return arr + (size_t)(gx + 8 * (k % NV) - alo[0]) + (size_t)an[0] * (size_t)(gy + 8 * (k / NV) - alo[1]);
    };
    const int fcomp = td.comp;

    // cells whose points can reach the tile, inside the patch's Lagrangian ghost box
    int clo[2], chi[2];
    bool any = true;
#pragma unroll
    for (int d = 0; d < 2; ++d)
    {
        clo[d] = max(flo[d] - a.reach, P.ilo[d] - a.idx_gcw);
        chi[d] = min(fhi[d] + a.reach, P.ihi[d] + a.idx_gcw);
        any = any && clo[d] <= chi[d];
    }
    // per-axis (bin, image offset) lists in increasing (bin, offset) order
    if (lane < 2)
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
    const int nx = __builtin_amdgcn_readfirstlane(s_ln[0]), ny = __builtin_amdgcn_readfirstlane(s_ln[1]);
    const int ncomb = nx * ny;
    // the lane's combination c of the canonical (y, x) order: its points and image code
    auto combination = [&](int c, int& st, int& ln, int& oc) IBAMR_INLINE {
        st = ln = oc = 0;
        if (c >= ncomb) return;
        const int kx = c % nx, ky = c / nx;
        const int m = bin_mem(2, s_lb[0][kx], s_lb[1][ky], 0, a.nb, a.nsb);
        st = a.bin_start[m];
        ln = a.bin_start[m + 1] - st;
        oc = (s_lo[0][kx] + 1) + 3 * (s_lo[1][ky] + 1);
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

    // the raw LEInteractor::spread adds each contribution to the existing value
    // (f.m4:1463); LDataManager::spread (interior mode) spreads into zeroed data and
    // adds the old values afterwards (LDataManager.cpp:594, 661-663)
    const bool from_old = a.mode == IBAMR_SPREAD_ACCUMULATE;
    double acc[NV * NV];
#pragma unroll
    for (int k = 0; k < NV * NV; ++k) acc[k] = from_old && in(k) ? (double)*at(k) : 0.0;

    const unsigned long long lt = (1ull << lane) - 1ull;
    const double vol = a.vol, rvol = a.rvol;
    int cb = -64, cq = 0, gtotal = 0, lex = 0;  // group, position in it, its points, the lane's first position
    int cf = 0;                                 // the combination holding the next position to fetch
    int nk = -1, noc = 4;
    int4 nc4 = make_int4(0, 0, 0, 0);
    double nX[2] = {0.0, 0.0};
    auto fetch = [&](int q0) IBAMR_INLINE {
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
        nc4 = a.cells[nk];
#pragma unroll
        for (int d = 0; d < 2; ++d) nX[d] = a.X[2 * (size_t)nk + d];
    };
    // the range of (X - x_lower) / dx - (flo - ilo) whose stencils reach the tile,
    // widened by what FP32 rounds
    const float tlo = (float)reach_lo<KER>() - 1e-3f;
    float thi[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) thi[d] = (float)(fhi[d] - flo[d]) + (float)reach_hi<KER>() + 1e-3f;
    bool more = true;
    int qh = 0, qn = 0;  // the ring's first entry and length
    for (;;)
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
                s_co[lane] = g_oc;
                __syncthreads();
                if (gtotal == 0) continue;
                fetch(0);
            }
            // the fetched candidates; the next ones' data are loaded meanwhile
            const int k = nk, oc = noc;
            const int cc[2] = {nc4.x, nc4.y};
            const int o[2] = {oc % 3 - 1, oc / 3 - 1};
            bool ok = k >= 0;
#pragma unroll
            for (int d = 0; d < 2; ++d)
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
                s_qo[p] = (unsigned char)oc;
            }
            qn += __popcll(m);
        }
        if (qn == 0) break;
        __syncthreads();
        const int n = min(qn, 64);
        // ---- stage them, one per lane
        int place = FAR | FAR << 8;  // (first x + 8) | (first y + 8) << 8, relative to the tile; bit 16: divide by vol
        if (lane < n)
        {
            const int q = (qh + lane) & (QCAP - 1);
            const int k = s_qk[q], oc = s_qo[q];
            const int o[2] = {oc % 3 - 1, oc / 3 - 1};
            T* r = s_row + lane * ROW;
            int b[2];
            T Fv = a.F[(size_t)a.fdepth * k + fcomp];
            const T fa = Fv < T(0) ? -Fv : Fv;
            // safe: div_by rounds the quotients by vol correctly
            bool safe = a.vol_div != 0 && (KT::IB || Fv == T(0) || (fa >= T(1e-30) && fa <= T(1e30)));
#pragma unroll
            for (int d = 0; d < 2; ++d)
            {
                // X + Xshift with Xshift = (double)(offset) * dx  (LIndexSetData.cpp:116)
                const double X = a.X[2 * (size_t)k + d];
                const double Xs = X + (double)(o[d] * a.pshift[d]) * a.dx[d];
                T w[W];
                if constexpr (FP64)
                {
                    b[d] = weights_1d_q<KER>(Xs, X, xl[d], a.dx[d], w, DivideBy{a.dx_ok ? a.rdx[d] : 0.0});
#pragma unroll
                    for (int i = 0; i < W; ++i)
                        if (!KT::IB || d == 1)
                            safe = safe && (w[i] == 0.0 || (fabs(w[i]) >= 1e-40 && fabs(w[i]) <= 1e40));
                    if (KT::IB && d == 1)  // IB folds 1/vol into w1 exactly as the reference
#pragma unroll
                        for (int i = 0; i < W; ++i) w[i] = safe ? div_by(w[i], vol, rvol) : w[i] / vol;
                }
                else
                    b[d] = weights_1d_u<KER>(Xs, X, xl[d], a.dx[d], w);
                b[d] += P.ilo[d] - flo[d];
#pragma unroll
                for (int i = 0; i < W; ++i) r[d * W + i] = w[i];
            }
            if (!FP64) Fv = Fv * T(rvol);
            r[2 * W] = Fv;
            if (b[0] > -W && b[0] < TILE && b[1] > -W && b[1] < TILE)
                place = (b[0] + 8) | (b[1] + 8) << 8 | (safe ? 0 : 1 << 16);
        }
        __syncthreads();
        // ---- apply them in order, four at a time: reads first, then the sums.  A lane
        // outside a stencil reads some weight and drops the product.
        for (int j = 0; j < n; j += 4)
        {
            double c[4];
            bool under[4];
            int which[4];  // of the lane's values the one that the stencil covers
            bool slow = false;
#pragma unroll
            for (int m = 0; m < 4; ++m)
            {
                const int jm = j + m;  // < 64
                const int pl = __builtin_amdgcn_readlane(place, jm);
                const int dx = x + 8 - (pl & 0xff), dy = y + 8 - ((pl >> 8) & 0xff);
                const int kx = NV == 2 && dx < 0 ? 1 : 0, ky = NV == 2 && dy < 0 ? 1 : 0;
                const unsigned ix = (unsigned)(dx + 8 * kx), iy = (unsigned)(dy + 8 * ky);
                which[m] = kx + NV * ky;
                under[m] = max(ix, iy) < (unsigned)W;
                slow = slow || (pl >> 16);
                const T* r = s_row + jm * ROW;
                const T wx = r[min(ix, (unsigned)(W - 1))], wy = r[W + min(iy, (unsigned)(W - 1))], Fj = r[2 * W];
                c[m] = (double)((wx * wy) * Fj);
            }
            if (FP64 && !KT::IB)  // ((w0*w1)*V)/vol
            {
                if (a.vol_div == 1)  // a power of two: the product rounds as the quotient does
                {
#pragma unroll
                    for (int m = 0; m < 4; ++m) c[m] = c[m] * rvol;
                }
                else if (!slow && a.vol_div == 2)
                {
#pragma unroll
                    for (int m = 0; m < 4; ++m) c[m] = div_by(c[m], vol, rvol);
                }
                else
                {
#pragma unroll
                    for (int m = 0; m < 4; ++m) c[m] = c[m] / vol;
                }
            }
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int k = 0; k < NV * NV; ++k) acc[k] = under[m] && which[m] == k ? acc[k] + c[m] : acc[k];
        }
        __syncthreads();
        qh = (qh + n) & (QCAP - 1);
        qn -= n;
    }
#pragma unroll
    for (int k = 0; k < NV * NV; ++k)
        if (in(k)) *at(k) = (overwrite || from_old) ? (T)acc[k] : (T)((double)*at(k) + acc[k]);
}
} // namespace
