// le_spread.hip -- the spread (LDataManager::spread inner loop,
// LDataManager.cpp:552-667 -> LEInteractor::spread -> lagrangian_<kernel>_spread{2,3}d):
// bin-order gather of the points, the spread kernels, the tile work list and its
// autotuner.
#include "le_plan_internal.h"

namespace ibamr
{
namespace
{
// Point data in bin order, so every later kernel reads slot k coalesced.
// Driven by the points: read X and F in the caller's order (coalesced) and
// write each point's record to its slot (a scattered write of a few bytes
// costs less than a scattered read of whole cache lines).
// ds (optional): F_ds[k][c] = F[k][c] * ds[k] (LDataManager.cpp:439-445).
template <typename T>
__global__ void k_scatter_points(const int* __restrict__ inv, int n, int ndim, const double* __restrict__ X,
                                 double* __restrict__ Xs, int fdepth, const T* __restrict__ F, T* __restrict__ Fs,
                                 const T* __restrict__ ds)
{
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= n) return;
    const size_t k = (size_t)inv[p];
    for (int d = 0; d < ndim; ++d) Xs[(size_t)ndim * k + d] = X[(size_t)ndim * p + d];
    if (F)
    {
        const T w = ds ? ds[p] : T(1);
        for (int c = 0; c < fdepth; ++c)
        {
            const T f = F[(size_t)fdepth * p + c];
            Fs[(size_t)fdepth * k + c] = ds ? f * w : f;
        }
    }
}

// FP32C 3-D spread set-up: for each point (bin order), axis d and variant v
// (v = 0: the level's x_lower; v = 1: x_lower - dx/2, the normal axis of side
// data, LEInteractor.cpp:3689) the first stencil index in the level's index
// space and the W weights, in the level's frame.  The spread's tiles then stage
// a candidate with loads instead of recomputing its weights for every tile it
// reaches; a patch or periodic image shifts the start by whole cells.  With
// perm, the kernel also performs the bin-order gather of X and F (side data:
// records of 3 positions and 3 force components, F times ds[p] when ds is
// given), so Xs is not read back.
template <int KER>
__global__ void k_point_weights(int n, double* __restrict__ Xs, int nvar, double3 xlo, double3 dx, int3 lo,
                                float* __restrict__ wt, int* __restrict__ st, const int* __restrict__ perm,
                                const double* __restrict__ Xin, const float* __restrict__ Fin,
                                float* __restrict__ Fs, const float* __restrict__ ds)
{
    constexpr int W = KernelTraits<KER>::W;
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const double xl[3] = {xlo.x, xlo.y, xlo.z}, h[3] = {dx.x, dx.y, dx.z};
    const int il[3] = {lo.x, lo.y, lo.z};
    double x[3];
    if (perm)
    {
        const size_t p = (size_t)perm[k];
        float f[3];
#pragma unroll
        for (int d = 0; d < 3; ++d)
        {
            x[d] = Xin[3 * p + d];
            f[d] = Fin[3 * p + d];
        }
        if (ds)  // F_ds[k][d] = F[k][d] * ds[k]  (LDataManager.cpp:439-445)
        {
            const float w = ds[p];
#pragma unroll
            for (int d = 0; d < 3; ++d) f[d] = f[d] * w;
        }
#pragma unroll
        for (int d = 0; d < 3; ++d)
        {
            Xs[3 * (size_t)k + d] = x[d];
            Fs[3 * (size_t)k + d] = f[d];
        }
    }
    else
#pragma unroll
        for (int d = 0; d < 3; ++d) x[d] = Xs[3 * (size_t)k + d];
#pragma unroll
    for (int d = 0; d < 3; ++d)
    {
        const double X = x[d];
        for (int v = 0; v < nvar; ++v)
        {
            float w[W];
            const int s0 = weights_1d<KER>(X, v ? xl[d] - 0.5 * h[d] : xl[d], h[d], w);
            const size_t row = (size_t)(d * nvar + v) * n + k;
            st[row] = il[d] + s0;
#pragma unroll
            for (int j = 0; j < W; ++j) wt[row * W + j] = w[j];
        }
    }
}

// FP32C 3-D: stencil starts and weights of the bin-ordered positions, used by
// the spread and the interpolation of the same positions
// (with X and F: the gather into bin order of side data's X and F as well)
template <int KER>
int launch_point_weights(ibamr_plan* P, hipStream_t s, const double* X = nullptr, const float* F = nullptr,
                         const float* ds = nullptr)
{
    if (!P->wt_d || !P->st_d) return fail(IBAMR_ERR_INVALID, "internal: no weight buffers");
    const int B = 256;
    hipLaunchKernelGGL((k_point_weights<KER>), dim3((P->npoints + B - 1) / B), dim3(B), 0, s, P->npoints, P->Xs_d,
                       P->nvar, make_double3(P->dom_xlo[0], P->dom_xlo[1], P->dom_xlo[2]),
                       make_double3(P->dx[0], P->dx[1], P->dx[2]),
                       make_int3(P->dom_lo[0], P->dom_lo[1], P->dom_lo[2]), P->wt_d, P->st_d,
                       X ? P->perm_d : nullptr, X, F, static_cast<float*>(P->Fs_d), ds);
    HIP_OK(hipGetLastError());
    return IBAMR_OK;
}

// ----------------------------------------------------------------------------- spread

template <typename T>
struct SpreadArgs
{
    const TileDesc* tiles;
    const PatchDev* patches;
    T* const* arrays;
    const double* X;   // positions in bin order (X[perm[k]] at slot k)
    const T* F;        // forces in bin order
    const int4* cells;
    const int* bin_start;
    int nb[3];
    int nsb[3];
    int bin;
    int dom_lo[3], dom_hi[3];
    int pshift[3];
    double dx[3];
    double rdx[3];  // 1 / dx; NaN for a dx out of div_by's range, which takes every position as near a tile
    int dx_ok;      // every dx in div_by's range
    double vol, rvol;
    int vol_div;   // FP64: 1: vol is a power of two, 2: quotients by vol from its reciprocal (div_by), 0: divisions
    int fdepth;
    int narr;
    int gcw[3];
    int idx_gcw;
    int reach;
    int side;
    int mode;
    // FP32C 3-D: the points' stencil starts and weights in the level's frame
    const float* wt;
    const int* st;
    int nvar;
    int npts;
};

} // namespace

#include "le_spread3d.h"
#include "le_spread2d.h"

namespace
{
template <typename T>
void fill_spread_args(const ibamr_plan* P, int slot, const void* F, const double* X, int mode, SpreadArgs<T>& a)
{
    a.patches = P->patches_d;
    a.arrays = reinterpret_cast<T* const*>(P->arrays_d[slot]);
    a.X = X;
    a.F = static_cast<const T*>(F);
    a.cells = P->cell_sorted_d;
    a.bin_start = P->bin_start_d;
    a.dx_ok = 1;
    for (int d = 0; d < 3; ++d)
    {
        a.nb[d] = P->nb[d];
        a.nsb[d] = P->nsb[d];
        a.dom_lo[d] = P->dom_lo[d];
        a.dom_hi[d] = P->dom_hi[d];
        a.pshift[d] = P->pshift[d];
        a.dx[d] = P->dx[d];
        a.rdx[d] = 1.0 / P->dx[d];
        if (P->dx[d] < 1e-60 || P->dx[d] > 1e60)
        {
            a.rdx[d] = std::numeric_limits<double>::quiet_NaN();
            a.dx_ok = 0;
        }
        a.gcw[d] = P->data_gcw[d];
    }
    a.bin = P->bin;
    a.vol = P->ndim == 3 ? (P->dx[0] * P->dx[1]) * P->dx[2] : P->dx[0] * P->dx[1];
    {
        int e;
        a.rvol = 1.0 / a.vol;
        a.vol_div = a.vol < 1e-60 || a.vol > 1e60 ? 0 : (std::frexp(a.vol, &e) == 0.5 ? 1 : 2);
    }
    a.fdepth = P->fdepth;
    a.narr = P->narr;
    a.idx_gcw = P->idx_gcw;
    a.reach = P->reach;
    a.side = P->centering == IBAMR_SIDE;
    a.mode = mode;
    a.wt = P->wt_d;
    a.st = P->st_d;
    a.nvar = P->nvar;
    a.npts = P->npoints;
}

// Spread tile shapes built for each form; the first is the default.
//   2-D: 16 x 16, taken as four 8 x 8 work items, or whole where few tiles have a point
//     (k_spread2, spread_list).
//   3-D: 8 x 8 or 16 x 4 grid lines (one per lane) times a column of z values
//     in registers (k_spread3b FP64, k_spread3 FP32C); an FP64 tile is cut along z
//     into work items (spread_cut).  FP32C keeps two register sets per z value (the
//     FP64 total and the chunk's FP32 partial), so its columns are shorter.
//     FP32C z extents of SWEEP_MIN_Z or more are z segments swept through a
//     register window (k_spread3s).
using Shape = std::array<int, 3>;
constexpr int SWEEP_MIN_Z = 48;
const std::vector<Shape>& tile_shapes(int ndim, int precision)
{
    static const std::vector<Shape> s2 = {{16, 16, 1}};
    static const std::vector<Shape> s64 = {{8, 8, 32}, {8, 8, 16}, {16, 4, 32}};
    static const std::vector<Shape> s32 = {{8, 8, 16}, {8, 8, 8}, {8, 8, 24}, {16, 4, 16},
                                           {8, 8, 64}, {8, 8, 128}, {8, 8, 256}};
    if (ndim == 2) return s2;
    return precision == IBAMR_FP64 ? s64 : s32;
}

// A shape is admissible when each axis of a tile reaches at most 16 (bin,
// image) entries (the image ranges partition the reachable cells, plus one
// split per domain side).  A z sweep takes up to S3S_MAXZ z entries and at
// most 64 (x, y) combinations per z layer, needs every stencil of a bin layer
// inside its register window (bin + 2 reach <= S3S_ZW) and the set-up pass's
// stencils (not computed for kernels whose stencil side depends on the
// unshifted X).
bool shape_admissible(const ibamr_plan* P, const Shape& sh)
{
    const bool sweep = P->ndim == 3 && sh[2] >= SWEEP_MIN_Z;
    if (sweep && (P->precision == IBAMR_FP64 || P->kernel == K_BS4 || P->kernel == K_BS6 ||
                  P->bin + 2 * P->reach > S3S_ZW))
        return false;
    int n[3] = {1, 1, 1};
    for (int d = 0; d < P->ndim; ++d)
    {
        n[d] = (sh[d] + 2 * P->reach + P->bin - 1) / P->bin + 3;
        if (n[d] > (sweep && d == 2 ? S3S_MAXZ : 16)) return false;
    }
    return !sweep || n[0] * n[1] <= 64;
}

// Tiles of the given extents over every array of every patch, of one depth component:
// spread_cut asks how many tiles share the points' work, and every component has the
// same points.
long count_tiles(const ibamr_plan* P, const Shape& ext)
{
    long total = 0;
    for (const PatchDev& pd : P->patches_h)
        for (int a = 0; a < P->narr; ++a)
        {
            long t = 1;
            for (int d = 0; d < P->ndim; ++d)
            {
                const int n = pd.ihi[d] - pd.ilo[d] + 1 + 2 * P->data_gcw[d] +
                              (P->centering == IBAMR_SIDE && d == a ? 1 : 0);
                t *= (n + ext[d] - 1) / ext[d];
            }
            total += t;
        }
    return total;
}

// z extent of a shape's work items (k_spread3b; the results do not depend on it).
// A wavefront takes its tile's points one after another, so the tiles along a
// dense surface are the critical path: 16 values each beat 32 everywhere (256^3
// IB_4, 10^6 points on a shell: 1.18 against 1.79 ms; AMR level of 384^3 0.79
// against 1.08 ms).  Fewer tiles than the GPU holds wavefronts (256 CUs x 16):
// 8 values (40^3, 432 tiles: 29 against 40 us; 64^3 IB_6, 1568 tiles: 259 against
// 357 us; at 8736 tiles 207 against 185 us; cell data of 8 components on 128^3, 2601
// tiles each, 200 k points on a shell 709 against 831 us, 20 k uniform 129 against 94).
// More than 128 tiles per SIMD: 24 for IB_4, IB_6 and BSPLINE_6, which then visit a
// point in fewer tiles (512^3 IB_6: 9.4 against 10.5 ms, IB_4 5.1 against 5.8,
// BSPLINE_6, 4.2 M points 7.9 against 9.0; at 86 k tiles IB_6 1.35 against 1.11 ms).
// The others keep 16 (512^3, 8.4 M points BSPLINE_3 5.8 against 6.6 ms; 4.2 M
// BSPLINE_4 4.6 against 5.1, BSPLINE_5 6.0 against 6.3; 2.1 M PIECEWISE_LINEAR 2.0
// against 2.2): more of their time goes into the tiles' own values.
int spread_cut(const ibamr_plan* P, const Shape& sh)
{
    if (P->ndim != 3 || P->precision != IBAMR_FP64) return sh[2];
    if (sh[0] != 8 || sh[2] != 32) return 16;
    if (count_tiles(P, {8, 8, 16}) < 4096) return 8;
    const bool tall = P->kernel == K_IB4 || P->kernel == K_IB6 || P->kernel == K_BS6;
    return tall && count_tiles(P, {8, 8, 24}) >= (1L << 17) ? 24 : 16;
}

// 2-D levels of at least this many 8 x 8 tiles also have a list of whole 16 x 16 tiles
// (spread_list).
constexpr long S2_MANY_TILES = 1L << 14;

// Work list of one tile shape: every tile of every array of every patch.
// XCD-aware launch order: workgroup i runs on XCD i % 8.  Tiles are grouped by
// (patch, z row, y row), each group holding that row of every array, and the
// groups are dealt to the XCDs in turn; each XCD runs its groups in (patch, z,
// y) order.  A group's tiles read the same point data through one L2 (all
// arrays, x neighbours), every XCD gets a share of every region (point clouds
// are rarely uniform, so contiguous eighths of the domain would leave some XCDs
// idle), and all XCDs sweep the domain together, so the data they re-read is
// recent in the shared last-level cache.
// Shapes cut into the same work items (FP64 8 x 8 x 32 and 8 x 8 x 16 where 32 is cut to
// 16) share one list.
int build_tiles(ibamr_plan* P, const Shape& sh, int cut, TileList& out)
{
    std::vector<TileDesc> tiles;
    const Shape ext = P->ndim == 3 ? Shape{sh[0], sh[1], cut} : Shape{cut, cut, 1};
    for (size_t i = 0; i < P->tlists.size() && &P->tlists[i] != &out; ++i)
    {
        const TileList& t = P->tlists[i];
        if (t.same < 0 && t.shape[0] == sh[0] && t.shape[1] == sh[1] && t.cut == cut)
        {
            out = t;
            out.same = (int)i;
            for (int d = 0; d < 3; ++d) out.shape[d] = sh[d];
            return IBAMR_OK;
        }
    }
    out.cut = cut;
    const int ncomp_tiles = P->centering == IBAMR_SIDE ? P->ndim : P->depth;
    std::vector<std::vector<TileDesc>> q(8);
    size_t g = 0;
    for (int i = 0; i < P->npatches; ++i)
    {
        const PatchDev& pd = P->patches_h[i];
        std::vector<std::array<int, 3>> nt(ncomp_tiles, std::array<int, 3>{1, 1, 1});
        int mt[3] = {1, 1, 1};
        for (int c = 0; c < ncomp_tiles; ++c)
        {
            const int axis = P->centering == IBAMR_SIDE ? c : -1;
            for (int d = 0; d < P->ndim; ++d)
            {
                const int n = pd.ihi[d] - pd.ilo[d] + 1 + 2 * P->data_gcw[d] + (d == axis ? 1 : 0);
                nt[c][d] = (n + ext[d] - 1) / ext[d];
                mt[d] = std::max(mt[d], nt[c][d]);
            }
        }
        for (int tz = 0; tz < mt[2]; ++tz)
            for (int ty = 0; ty < mt[1]; ++ty, ++g)
                for (int c = 0; c < ncomp_tiles; ++c)
                    if (ty < nt[c][1] && tz < nt[c][2])
                        for (int tx = 0; tx < nt[c][0]; ++tx) q[g % 8].push_back(TileDesc{i, c, {tx, ty, tz}});
    }
    size_t per = 0;
    for (const auto& v : q) per = std::max(per, v.size());
    tiles.assign(8 * per, TileDesc{-1, 0, {0, 0, 0}});
    for (int x = 0; x < 8; ++x)
        for (size_t k = 0; k < q[x].size(); ++k) tiles[8 * k + x] = q[x][k];
    out.n = (int)tiles.size();
    for (int d = 0; d < 3; ++d) out.shape[d] = sh[d];
    HIP_OK(hipMalloc(&out.d, sizeof(TileDesc) * std::max<size_t>(1, tiles.size())));
    if (!tiles.empty()) HIP_OK(hipMemcpy(out.d, tiles.data(), sizeof(TileDesc) * tiles.size(), hipMemcpyHostToDevice));
    return IBAMR_OK;
}

// The work list a spread takes: the one chosen, or its pieces of 8 where the autotuner
// found them faster; but for few points per tile
//   IB_4 3-D, fewer than two per tile of 24 values, overwriting: the list of 16 values:
//     most tiles then write zeros, and those of IB_4 run four to a SIMD, whose
//     unfinished lines of 24 planes no longer fit the L2 (512^3, 20000 points: 1.33 ms,
//     0.93 with 16 values; 10^6 points 1.36 and 1.35; accumulating 0.31 and 0.37).
//   2-D, fewer than t^1.5 / 1024 at t tiles of 8 x 8 (1536 where an empty tile's values
//     are not touched): whole 16 x 16 tiles, a quarter of the workgroups, since the
//     launch and an empty tile's own steps are what it costs (FP64 IB_4, side: 2048^2,
//     5000 points 45 against 95 us uniform, 34 against 77 on a circle; 4096^2, 20000 in
//     a disc 126 against 321, 2 x 10^5 on a circle 224 against 312).  With more points
//     the longest chain decides, and a 16 x 16 tile's is up to four times as long.
//     Workgroups grow with t, the chain of points on a curve with their number over
//     t^0.5, so the line is at t^1.5: 800^2, 3000 on a circle 17 against 19, 1400^2,
//     10^4 34 and 41, 3 x 10^4 68 and 53; 2048^2, 6 x 10^4 99 and 91 (uniform 64 and
//     141).  Accumulating 2048^2, 45000 on a circle 74 and 63, 5000 23 and 49.
const TileList& spread_list(const ibamr_plan* P, int mode)
{
    const TileList& tl = P->tlists[P->tcur];
    if (P->ndim == 2)
    {
        const double n = P->npoints, t = tl.n;
        const double line = t * std::sqrt(t) / (mode == IBAMR_SPREAD_OVERWRITE ? 1024 : 1536);
        return P->tsparse.n > 0 && n < line ? P->tsparse : tl;
    }
    if (P->fine && (P->tcur == 0 || tl.same == 0)) return P->tfine;
    if (P->kernel == K_IB4 && P->precision == IBAMR_FP64 && mode == IBAMR_SPREAD_OVERWRITE && tl.cut == 24 &&
        P->npoints < 2L * tl.n)
        for (const TileList& t : P->tlists)
            if (t.shape[0] == 8 && t.cut == 16) return t;
    return tl;
}

int find_shape(const ibamr_plan* P, const int* shape)
{
    for (size_t i = 0; i < P->tlists.size(); ++i)
        if (P->tlists[i].shape[0] == shape[0] && P->tlists[i].shape[1] == shape[1] &&
            P->tlists[i].shape[2] == shape[2])
            return (int)i;
    return -1;
}
} // namespace

int build_tile_lists(ibamr_plan* P)
{
    for (const Shape& sh : tile_shapes(P->ndim, P->precision))
    {
        if (!shape_admissible(P, sh)) continue;
        P->tlists.emplace_back();
        const int rc = build_tiles(P, sh, P->ndim == 3 ? spread_cut(P, sh) : S2_TILE, P->tlists.back());
        if (rc != IBAMR_OK) return rc;
        if (P->ndim == 2 && P->tlists.back().n >= S2_MANY_TILES)
        {
            const int rc2 = build_tiles(P, sh, 2 * S2_TILE, P->tsparse);
            if (rc2 != IBAMR_OK) return rc2;
        }
    }
    if (P->tlists.empty()) return fail(IBAMR_ERR_INVALID, "drift_cells too large for the tile size");
    P->tcur = 0;
    return IBAMR_OK;
}
} // namespace ibamr

extern "C" {

int ibamr_plan_spread(ibamr_plan* P, int slot, const void* F, const double* X, int mode, void* stream)
{
    return ibamr_plan_spread_ds(P, slot, F, X, nullptr, mode, stream);
}

int ibamr_plan_spread_ds(ibamr_plan* P, int slot, const void* F, const double* X, const void* ds, int mode,
                         void* stream)
{
    if (!P) return fail(IBAMR_ERR_INVALID, "null plan");
    if (slot < 0 || slot >= MAX_SLOTS || !P->arrays_d[slot]) return fail(IBAMR_ERR_INVALID, "slot not bound");
    if (P->npoints < 0) return fail(IBAMR_ERR_NOT_BINNED, "points not binned");
    if (mode != IBAMR_SPREAD_ACCUMULATE && mode != IBAMR_SPREAD_OVERWRITE && mode != IBAMR_SPREAD_ACCUMULATE_INTERIOR)
        return fail(IBAMR_ERR_INVALID, "bad mode");
    if (P->npoints > 0 && (!F || !X)) return fail(IBAMR_ERR_INVALID, "null F or X");
    if (P->tlists.empty() || P->tlists[P->tcur].n == 0) return IBAMR_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    return dispatch(P->ndim, P->kernel, P->precision, [&](auto nd, auto ker, auto prec) -> int {
        using T = decltype(prec);
        constexpr int NDIM = decltype(nd)::value;
        constexpr int KER = decltype(ker)::value;
        SpreadArgs<T> a{};
        fill_spread_args<T>(P, slot, F, X, mode, a);
        const TileList& tl = spread_list(P, mode);
        a.tiles = tl.d;
        if (P->npoints > 0)
        {
            const int B = 256;
            // FP32C 3-D: stencils set up here (not for kernels whose side depends on the unshifted X)
            constexpr bool WTS = NDIM == 3 && sizeof(T) == 4 && !side_by_unshifted_x<KER>();
            if constexpr (WTS)
            {
                if (P->fdepth == NDIM)
                {
                    // gather (with F*ds) and stencils in one pass
                    const int rc = launch_point_weights<KER>(P, s, X, reinterpret_cast<const float*>(F),
                                                             reinterpret_cast<const float*>(ds));
                    if (rc != IBAMR_OK) return rc;
                }
            }
            if (!WTS || P->fdepth != NDIM)
            {
                // the points in bin order
                if (P->fdepth == NDIM)
                    hipLaunchKernelGGL((k_gather_points<NDIM, T>), dim3((P->npoints + B - 1) / B), dim3(B), 0, s,
                                       P->perm_d, P->npoints, X, P->Xs_d, static_cast<const T*>(F),
                                       static_cast<T*>(P->Fs_d), static_cast<const T*>(ds));
                else
                    hipLaunchKernelGGL(k_scatter_points<T>, dim3((P->npoints + B - 1) / B), dim3(B), 0, s, P->idx_d,
                                       P->npoints, NDIM, X, P->Xs_d, P->fdepth, static_cast<const T*>(F),
                                       static_cast<T*>(P->Fs_d), static_cast<const T*>(ds));
                HIP_OK(hipGetLastError());
                if constexpr (WTS)
                {
                    const int rc = launch_point_weights<KER>(P, s);
                    if (rc != IBAMR_OK) return rc;
                }
            }
            P->xs_valid = true;
            P->ws_valid = WTS;
        }
        a.X = P->Xs_d;
        a.F = static_cast<const T*>(P->Fs_d);
        if (!a.tiles || !a.patches || !a.arrays || !a.X || !a.F || !a.cells || !a.bin_start)
            return fail(IBAMR_ERR_INVALID, "internal: incomplete spread arguments");
        hipEvent_t t_end;
        const int trc = time_begin(P, 0, s, &t_end);
        if (trc != IBAMR_OK) return trc;
        if constexpr (NDIM == 3)
        {
            const dim3 G(tl.n), B(64);
#define IBAMR_S3(TX, ZC)                                                              \
    if (tl.shape[0] == TX && tl.shape[2] == ZC)                                       \
    {                                                                                 \
        hipLaunchKernelGGL((k_spread3<KER, ZC, TX>), G, B, 0, s, a);                  \
        HIP_OK(hipGetLastError());                                                    \
        if (t_end) HIP_OK(hipEventRecord(t_end, s));                                  \
        return IBAMR_OK;                                                              \
    }
            if constexpr (sizeof(T) == 8)
            {
#define IBAMR_S3B(TX, ZC)                                                      \
    if (tl.shape[0] == TX && tl.cut == ZC)                                     \
    {                                                                          \
        hipLaunchKernelGGL((k_spread3b<KER, ZC, TX>), G, B, 0, s, a);          \
        HIP_OK(hipGetLastError());                                             \
        if (t_end) HIP_OK(hipEventRecord(t_end, s));                           \
        return IBAMR_OK;                                                       \
    }
                IBAMR_S3B(8, 24)
                IBAMR_S3B(8, 16)
                IBAMR_S3B(8, 8)
                IBAMR_S3B(16, 16)
#undef IBAMR_S3B
            }
            else
            {
                IBAMR_S3(8, 16)
                IBAMR_S3(8, 8)
                IBAMR_S3(8, 24)
                IBAMR_S3(16, 16)
                if constexpr (!side_by_unshifted_x<KER>())
                    if (tl.shape[0] == 8 && tl.shape[2] >= SWEEP_MIN_Z)
                    {
                        if (P->npoints > 0 && !P->ws_valid)
                            return fail(IBAMR_ERR_INVALID, "internal: z sweep without stencils");
                        hipLaunchKernelGGL((k_spread3s<KER, 8>), G, B, 0, s, a, tl.shape[2]);
                        HIP_OK(hipGetLastError());
                        if (t_end) HIP_OK(hipEventRecord(t_end, s));
                        return IBAMR_OK;
                    }
            }
#undef IBAMR_S3
            return fail(IBAMR_ERR_INVALID, "internal: tile shape without a kernel");
        }
        else
        {
            const auto kernel = tl.cut == S2_TILE ? k_spread2<KER, T, 1> : k_spread2<KER, T, 2>;
            hipLaunchKernelGGL(kernel, dim3(tl.n), dim3(64), 0, s, a);
        }
        HIP_OK(hipGetLastError());
        if (t_end) HIP_OK(hipEventRecord(t_end, s));
        return IBAMR_OK;
    });
}

int ibamr_plan_set_tile_shape(ibamr_plan* P, const int* shape)
{
    if (!P || !shape) return fail(IBAMR_ERR_INVALID, "null argument");
    const int i = find_shape(P, shape);
    if (i < 0)
        return fail(IBAMR_ERR_INVALID, "tile shape " + std::to_string(shape[0]) + "x" + std::to_string(shape[1]) + "x" +
                                           std::to_string(shape[2]) + " not built for this plan");
    P->tcur = i;
    return IBAMR_OK;
}

int ibamr_plan_get_tile_shape(const ibamr_plan* P, int* shape)
{
    if (!P || !shape) return fail(IBAMR_ERR_INVALID, "null argument");
    for (int d = 0; d < 3; ++d) shape[d] = P->tlists.empty() ? 0 : P->tlists[P->tcur].shape[d];
    return IBAMR_OK;
}

int ibamr_plan_set_tile_height(ibamr_plan* P, int height)
{
    if (!P) return fail(IBAMR_ERR_INVALID, "null plan");
    for (size_t i = 0; i < P->tlists.size(); ++i)
        if (P->tlists[i].shape[2] == height)
        {
            P->tcur = (int)i;
            return IBAMR_OK;
        }
    return fail(IBAMR_ERR_INVALID, "tile height " + std::to_string(height) + " not built for this plan");
}

int ibamr_plan_get_tile_height(const ibamr_plan* P, int* height)
{
    if (!P || !height) return fail(IBAMR_ERR_INVALID, "null argument");
    *height = P->tlists.empty() ? 0 : P->tlists[P->tcur].shape[2];
    return IBAMR_OK;
}

int ibamr_plan_autotune(ibamr_plan* P, int slot, const void* F, const double* X, int reps, int* shapes, float* ms,
                        int* ncand, void* stream)
{
    if (!P || !shapes || !ms || !ncand) return fail(IBAMR_ERR_INVALID, "null argument");
    if (P->npoints < 0) return fail(IBAMR_ERR_NOT_BINNED, "points not binned");
    *ncand = 0;
    if ((int)P->tlists.size() > IBAMR_MAX_TILE_SHAPES) return fail(IBAMR_ERR_INVALID, "internal: too many tile shapes");
    reps = std::max(1, reps);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool timing = P->timing;
    P->timing = false;  // the trials are not the caller's launches
    const int start = P->tcur;
    const bool start_fine = P->fine;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int best = start;
    float best_ms = std::numeric_limits<float>::infinity();
    // rounds over all shapes, each timing `reps` spreads per shape; a shape's
    // time is its fastest round (the shapes are interleaved, so a slow spell of
    // the device does not fall on one shape only)
    constexpr int ROUNDS = 3;
    auto run = [&]() -> int {
        HIP_OK(hipEventCreate(&e0));
        HIP_OK(hipEventCreate(&e1));
        const size_t ns = P->tlists.size();
        // FP64 3-D: the default shape is also tried in pieces of 8 values, whose shorter
        // chains pay on crowded surfaces (131^3, 2.1 M points on a shell: IB_6 8.0 against
        // 10.6 ms in pieces of 16, IB_4 4.8 against 7.0; spread over the volume 10 to 24 %
        // slower): two sets of points that no rule on sizes tells apart.
        const bool fine = P->ndim == 3 && P->precision == IBAMR_FP64 && P->tlists[0].shape[0] == 8 && P->tlists[0].cut > 8;
        if (fine && !P->tfine.d)
        {
            const int* sh = P->tlists[0].shape;
            const int r = build_tiles(P, Shape{sh[0], sh[1], sh[2]}, 8, P->tfine);
            if (r != IBAMR_OK)
            {
                if (P->tfine.d) (void)hipFree(P->tfine.d);  // not written: the next call builds it anew
                P->tfine = TileList();
                return r;
            }
        }
        float fine_ms = std::numeric_limits<float>::infinity();
        auto trial = [&](size_t i, int n) -> int {  // i = ns: the default shape in pieces of 8
            P->fine = i == ns;
            P->tcur = i == ns ? 0 : (int)i;
            for (int k = 0; k < n; ++k)
            {
                const int r = ibamr_plan_spread(P, slot, F, X, IBAMR_SPREAD_OVERWRITE, stream);
                if (r != IBAMR_OK) return r;
            }
            return IBAMR_OK;
        };
        auto skip = [&](size_t i) { return i == ns ? !fine : P->tlists[i].same >= 0; };
        for (size_t i = 0; i <= ns; ++i)
        {
            if (i < ns)
            {
                for (int d = 0; d < 3; ++d) shapes[3 * i + d] = P->tlists[i].shape[d];
                ms[i] = std::numeric_limits<float>::infinity();
            }
            if (skip(i)) continue;
            const int r = trial(i, 1);  // untimed
            if (r != IBAMR_OK) return r;
        }
        for (int round = 0; round < ROUNDS; ++round)
            for (size_t i = 0; i <= ns; ++i)
            {
                if (skip(i)) continue;
                HIP_OK(hipEventRecord(e0, s));
                const int r = trial(i, reps);
                if (r != IBAMR_OK) return r;
                HIP_OK(hipEventRecord(e1, s));
                HIP_OK(hipEventSynchronize(e1));
                float t = 0.0f;
                HIP_OK(hipEventElapsedTime(&t, e0, e1));
                float& m = i == ns ? fine_ms : ms[i];
                m = std::min(m, t / reps);
            }
        P->fine = fine_ms < ms[0];
        ms[0] = std::min(ms[0], fine_ms);
        for (size_t i = 0; i < ns; ++i)  // a shared list has its owner's time
            if (P->tlists[i].same >= 0) ms[i] = ms[P->tlists[i].same];
        for (size_t i = 0; i < ns; ++i)
            if (ms[i] < best_ms)
            {
                best_ms = ms[i];
                best = (int)i;
            }
        return IBAMR_OK;
    };
    const int rc = run();
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    P->timing = timing;
    if (rc != IBAMR_OK)
    {
        P->tcur = start;
        P->fine = start_fine;
        return rc;
    }
    *ncand = (int)P->tlists.size();
    P->tcur = best;
    return IBAMR_OK;
}

} // extern "C"
