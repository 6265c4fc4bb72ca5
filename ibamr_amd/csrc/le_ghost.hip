// le_ghost.hip -- grid steps around the path: periodic and same-level
// ghost fills (the RefineSchedule fill before interp, LDataManager.cpp:742-745) and
// the physical-boundary Robin operators (CartCell/CartSideRobinPhysBdryOp).
#include "le_plan_internal.h"

namespace ibamr
{
namespace
{
// ----------------------------------------------------------------------------- periodic ghost fill

// Periodic ghost fill of one array of a single-patch, fully periodic level:
// every value outside the core [g, g+N) of each axis takes the value of its
// periodic image, which lies in the core (the ghost width never exceeds the
// period).  Only the ghost shell is enumerated: z slabs (whole planes), then y
// slabs inside the core z range, then x slabs inside the core y and z ranges.
// One launch fills every array and component of the level (blockIdx.y): a 2-D or
// small 3-D fill is a few microseconds of launch and latency, not of copying.
struct PeriodicArgs
{
    void* arr[3];
    int n[3][3];      // extents of each array
    long sz[3], sy[3], sx[3];
    int g[3], N[3];
    int ncomps;
};

template <typename T, typename I>
__global__ void k_fill_periodic(PeriodicArgs a)
{
    const int ai = blockIdx.y / a.ncomps;
    const int n0 = a.n[ai][0], n1 = a.n[ai][1], n2 = a.n[ai][2];
    const int g0 = a.g[0], g1 = a.g[1], g2 = a.g[2], N0 = a.N[0], N1 = a.N[1], N2 = a.N[2];
    T* __restrict__ arr = static_cast<T*>(a.arr[ai]) + (size_t)(blockIdx.y % a.ncomps) * n0 * n1 * n2;
    I t = (I)blockIdx.x * blockDim.x + threadIdx.x;  // I holds every shell index and the launch's round-up
    const I sz = (I)a.sz[ai], sy = (I)a.sy[ai], sx = (I)a.sx[ai];
    int i0, i1, i2;
    if (t < sz)
    {
        const I plane = (I)n0 * n1;
        const int q = (int)(t / plane);                       // which ghost plane
        const I r = t - (I)q * plane;
        i2 = q < g2 ? q : q - g2 + g2 + N2;                   // lower planes, then upper planes
        i1 = (int)(r / (I)n0);
        i0 = (int)(r - (I)i1 * n0);
    }
    else if ((t -= sz) < sy)
    {
        const I slab = (I)(n1 - N1) * n0;                    // per core z plane
        const int z = (int)(t / slab);
        const I r = t - (I)z * slab;
        const int q = (int)(r / (I)n0);
        i0 = (int)(r - (I)q * n0);
        i1 = q < g1 ? q : q - g1 + g1 + N1;
        i2 = g2 + z;
    }
    else if ((t -= sy) < sx)
    {
        const I w = (I)(n0 - N0);                            // per core (y, z) row
        const I row = t / w;
        const int q = (int)(t - row * w);
        i0 = q < g0 ? q : q - g0 + g0 + N0;
        i1 = g1 + (int)(row % (I)N1);
        i2 = g2 + (int)(row / (I)N1);
    }
    else
        return;
    int j0 = i0 - g0, j1 = i1 - g1, j2 = i2 - g2;
    j0 += j0 < 0 ? N0 : (j0 >= N0 ? -N0 : 0);
    j1 += j1 < 0 ? N1 : (j1 >= N1 ? -N1 : 0);
    j2 += j2 < 0 ? N2 : (j2 >= N2 ? -N2 : 0);
    arr[(long)i0 + (long)n0 * (i1 + (long)n1 * i2)] =
        arr[(long)(j0 + g0) + (long)n0 * ((j1 + g1) + (long)n1 * (j2 + g2))];
}

// Same-level ghost fill (the RefineSchedule::fillData step before interp,
// LDataManager.cpp:742-745, restricted to copies between patches of one level):
// every ghost value of every patch array whose index -- wrapped across periodic
// directions -- lies in another patch's (or, periodically, its own) interior
// side box is copied from there.  Ghost values outside the domain of a
// non-periodic direction, or not covered by the level (coarse-fine boundary),
// are left as they are.
constexpr int FILL_SEG = 1024;  // values of a slab per workgroup

template <typename T>
struct FillArgs
{
    const int4* segs;
    const PatchDev* patches;
    T* const* arrays;
    const int* bin_patch_start;
    const int* bin_patches;
    int narr, side, depth;
    int gcw[3];
    int dom_lo[3], dom_hi[3];
    int pshift[3];
    int nb[3], nsb[3];
    int bin;
};

// Ghost values are enumerated slab by slab of a patch array's ghost shell (the
// interior is never visited), FILL_SEG of a slab per workgroup: segs holds
// (patch, array, slab, first value of the slab); slab 2 d + u lies outside the
// interior of axis d on its lower (u = 0) or upper side, inside the interior of
// the axes above d, and covers the whole array along the axes below d.
// Bound by the lookups (bin -> patches -> box, cached) and 24-byte rows of the x
// slabs.  Level of 229 patches (edges 16-64) around shells in 512^3, ghost width 3,
// FP32: 300 us, 2241 us when every array value was visited with 64-bit indices.
template <int NDIM, typename T>
__global__ __launch_bounds__(256) void k_fill_level(FillArgs<T> a)
{
    const int4 sg = a.segs[blockIdx.x];
    const int pid = sg.x, arr_i = sg.y, slab = sg.z;
    const int axis = a.side ? arr_i : -1;
    const PatchDev& P = a.patches[pid];
    int n[3] = {1, 1, 1}, lo[3] = {0, 0, 0};     // the array's extents and lower index
    int s0[3] = {0, 0, 0}, sn[3] = {1, 1, 1};    // the slab's first array index and extents
#pragma unroll
    for (int d = 0; d < NDIM; ++d)
    {
        lo[d] = P.ilo[d] - a.gcw[d];
        n[d] = P.ihi[d] - P.ilo[d] + 1 + 2 * a.gcw[d] + (d == axis ? 1 : 0);
        s0[d] = (slab >> 1) < d ? a.gcw[d] : 0;
        sn[d] = n[d] - 2 * s0[d];
        if ((slab >> 1) == d)
        {
            s0[d] = (slab & 1) ? n[d] - a.gcw[d] : 0;
            sn[d] = a.gcw[d];
        }
    }
    const int count = sn[0] * sn[1] * sn[2];
    T* __restrict__ dst = a.arrays[pid * a.narr + arr_i];
    const size_t ptot = (size_t)n[0] * n[1] * n[2];
    const int ncomp = a.side ? 1 : a.depth;
    const int end = min(count, sg.w + FILL_SEG);
    for (int e = sg.w + (int)threadIdx.x; e < end; e += 256)
    {
        const unsigned r = (unsigned)e / (unsigned)sn[0];
        const int idx[3] = {s0[0] + (int)((unsigned)e - r * (unsigned)sn[0]), s0[1] + (int)(r % (unsigned)sn[1]),
                            s0[2] + (int)(r / (unsigned)sn[1])};
        int w[3] = {0, 0, 0};
        bool ok = true;
#pragma unroll
        for (int d = 0; d < NDIM; ++d)
        {
            const int i = lo[d] + idx[d];
            const int N = a.pshift[d];
            if (N > 0)
            {
                // a few periods at most: the ghost width never exceeds one
                w[d] = i;
                while (w[d] < a.dom_lo[d]) w[d] += N;
                while (w[d] >= a.dom_lo[d] + N) w[d] -= N;
            }
            else
            {
                // beyond a physical boundary: not filled here
                ok = ok && i >= a.dom_lo[d] && i <= a.dom_hi[d] + (d == axis ? 1 : 0);
                w[d] = i;
            }
        }
        if (!ok) continue;
        // owner: a patch whose interior side box holds the wrapped index; its cell,
        // or for a side axis also the cell below (the face is that cell's upper face)
        int q = -1;
        for (int tries = 0; tries < (axis < 0 ? 1 : 2) && q < 0; ++tries)
        {
            int b[3] = {0, 0, 0};
            bool in_dom = true;
#pragma unroll
            for (int d = 0; d < NDIM; ++d)
            {
                const int c = w[d] - (tries == 1 && d == axis ? 1 : 0);
                in_dom = in_dom && c >= a.dom_lo[d] && c <= a.dom_hi[d];
                b[d] = (int)((unsigned)(c - a.dom_lo[d]) / (unsigned)a.bin);
            }
            if (!in_dom) continue;
            const int key = bin_mem(NDIM, b[0], b[1], b[2], a.nb, a.nsb);
            for (int j = a.bin_patch_start[key]; j < a.bin_patch_start[key + 1] && q < 0; ++j)
            {
                const int cand = a.bin_patches[j];
                const PatchDev& Q = a.patches[cand];
                bool in = true;
#pragma unroll
                for (int d = 0; d < NDIM; ++d)
                    in = in && w[d] >= Q.ilo[d] && w[d] <= Q.ihi[d] + (d == axis ? 1 : 0);
                if (in) q = cand;
            }
        }
        if (q < 0) continue;  // not covered by this level
        const PatchDev& Q = a.patches[q];
        size_t src = 0, stride = 1;
#pragma unroll
        for (int d = 0; d < NDIM; ++d)
        {
            src += stride * (size_t)(w[d] - (Q.ilo[d] - a.gcw[d]));
            stride *= (size_t)(Q.ihi[d] - Q.ilo[d] + 1 + 2 * a.gcw[d] + (d == axis ? 1 : 0));
        }
        const T* __restrict__ from = a.arrays[q * a.narr + arr_i];
        const size_t at = (size_t)idx[0] + (size_t)n[0] * ((size_t)idx[1] + (size_t)n[1] * (size_t)idx[2]);
        for (int cd = 0; cd < ncomp; ++cd) dst[(size_t)cd * ptot + at] = from[(size_t)cd * stride + src];
    }
}
} // namespace

// ----------------------------------------------------------------------------- physical boundary

namespace
{
// The LINEAR Robin ghost operators of CartCellRobinPhysBdryOp / CartSideRobinPhysBdryOp
// (cartphysbdryop{2,3}d.f.m4), adjoint (accumulateFromPhysicalBoundaryData) and
// forward (setPhysicalBoundaryConditions).  The reference applies the operators of
// a patch one after another; every operator updates one component.  Here operators
// of one component whose index regions do not meet run together (a stage, one
// launch over all patches; stages in the reference's order, bdry_stages), and
// inside an operator every thread owns values that no other thread updates, taking
// their updates in the reference's order from registers.  So every value sees the
// reference's sequence of operations.
// Bound by launches and latency (a boundary layer is small): 160 x 144 x 200 box,
// 8 patches, ghost width 3, side FP64: 72 us per pass in six launches, 1933 us when
// one workgroup walked a patch's operators, each update waiting for memory.
enum BdryKind : int
{
    B_CC_FACE = 0,   // cell data, codim 1 (also side data's transverse components)
    B_SC_FACE,       // side data, codim 1, normal component
    B_CC_EDGE,       // cell data, 3-D codim 2
    B_CC_CORNER,     // cell data, codim ndim
    B_SC_EDGE,       // side data, 3-D codim 2, one of its two components
    B_SC_CORNER      // side data, codim ndim, one component
};

template <typename T>
struct BdryArgs
{
    const BdryOp* ops;
    const int2* blocks;  // (operator, first work item) per workgroup of this stage
    const int* boxes;
    // Robin coefficients of codim-1 boxes: for box slot k and coefficient array j
    // (an axis of side data, a component of cell data), a, b and g over the box's
    // columns start at coef + coef_off[k * m + j], m = ndim (side) or depth (cell)
    const double* coef;
    const long* coef_off;
    const PatchDev* patches;
    T* const* arrays;
    int ndim, side, depth, narr, gcw, adjoint;
    double dx[3];
};

template <typename T>
struct BPatch
{
    int ndim, side, gcw;
    int ilo[3], ihi[3];
    long vol;  // values per depth component (cell data)
    T* arr[3];
    __device__ T* at(int a, int comp, const int* x) const
    {
        long off = 0, mul = 1;
        for (int d = 0; d < ndim; ++d)
        {
            const int n = ihi[d] - ilo[d] + 1 + 2 * gcw + ((side && d == a) ? 1 : 0);
            off += (long)(x[d] - (ilo[d] - gcw)) * mul;
            mul *= n;
        }
        return side ? arr[a] + off : arr[0] + (long)comp * vol + off;
    }
};

__device__ inline int bp_tangential_dev(int ndim, int dir, int* t)
{
    int m = 0;
    for (int d = ndim - 1; d >= 0; --d)
        if (d != dir) t[m++] = d;
    return m;
}

// column c of a face: coordinates of the tangential dims
__device__ inline void face_column(int ndim, int dir, const int* blo, const int* bhi, long c, int* x)
{
    int t[2];
    const int nt = bp_tangential_dev(ndim, dir, t);
    const int n_in = bhi[t[nt - 1]] - blo[t[nt - 1]] + 1;
    x[t[nt - 1]] = blo[t[nt - 1]] + (int)(c % n_in);
    if (nt > 1) x[t[0]] = blo[t[0]] + (int)(c / n_in);
}

__device__ inline long face_columns(int ndim, int dir, const int* blo, const int* bhi)
{
    long m = 1;
    for (int d = 0; d < ndim; ++d)
        if (d != dir) m *= (long)(bhi[d] - blo[d] + 1);
    return m;
}

// codim 1, cell data and side data's transverse components: work item (column,
// layer i): ghost layer i and its mirror layer, which no other item touches
template <typename T>
__device__ void bd_cc_face(const BPatch<T>& P, int a, int comp, int loc, int dhi, const int* blo, const int* bhi,
                           const double* cf, int adjoint, const double* dx, long t)
{
    const int ndim = P.ndim, dir = loc / 2, lower = (loc % 2) == 0;
    const double h = dx[loc / ndim];  // as the Fortran indexes it
    const int sgn = lower ? -1 : 1;
    const int ig = lower ? P.ilo[dir] - 1 : dhi + 1, ii = lower ? P.ilo[dir] : dhi;
    const long ncol = face_columns(ndim, dir, blo, bhi);
    const long c = t % ncol;
    const int i = (int)(t / ncol);
    int x[3] = {0, 0, 0};
    face_column(ndim, dir, blo, bhi, c, x);
    // column c of the coefficient box (the lower tangential axis fastest, as acoef(j,k))
    const double ca = cf[c], cb = cf[ncol + c], cg = cf[2 * ncol + c];
    const double n = 1.0 + 2.0 * i;
    const double f_i = -(ca * n * h - 2.0 * cb) / (ca * n * h + 2.0 * cb);
    const double f_g = 2.0 * n * h / (ca * n * h + 2.0 * cb);
    int xg[3] = {x[0], x[1], x[2]}, xi[3] = {x[0], x[1], x[2]};
    xg[dir] = ig + sgn * i;
    xi[dir] = ii - sgn * i;
    T* g = P.at(a, comp, xg);
    T* v = P.at(a, comp, xi);
    if (adjoint)
        *v = (T)((double)*v + f_i * (double)*g);
    else
        *g = (T)(f_i * (double)*v + f_g * cg);
}

// codim 1, side data's normal component: the boundary face of a column collects
// from every layer, so the adjoint's work item is a column; the forward's (column,
// layer)
template <typename T>
__device__ void bd_sc_face(const BPatch<T>& P, int loc, const int* blo, const int* bhi, const double* cf, int adjoint,
                           const double* dx, long t)
{
    const int ndim = P.ndim, dir = loc / 2, lower = (loc % 2) == 0;
    const double h = dx[loc / ndim];
    const int sgn = lower ? -1 : 1;
    const int ib = lower ? P.ilo[dir] : P.ihi[dir] + 1;
    const long ncol = face_columns(ndim, dir, blo, bhi);
    const long c = t % ncol;
    int x[3] = {0, 0, 0};
    face_column(ndim, dir, blo, bhi, c, x);
    const double ca = cf[c], cb = cf[ncol + c], cg = cf[2 * ncol + c];
    const bool dirichlet = fabs(cb) < 1.0e-12;  // per face (scrobinphysbdryop1: abs(b) .lt. 1.d-12)
    int xb[3] = {x[0], x[1], x[2]};
    xb[dir] = ib;
    T* ub = P.at(dir, 0, xb);
    auto factors = [&](int i, double& f_i, double& f_b, double& f_g) {
        f_i = -1.0, f_b = 2.0, f_g = 0.0;
        if (!dirichlet)
        {
            const double n = 2.0 * i;
            f_i = 1.0;
            f_b = -ca * n * h / cb;
            f_g = n * h / cb;
        }
    };
    int xg[3] = {x[0], x[1], x[2]}, xi[3] = {x[0], x[1], x[2]};
    double f_i, f_b, f_g;
    if (!adjoint)
    {
        const int i = 1 + (int)(t / ncol);
        const double u_b = dirichlet ? cg / ca : (double)*ub;
        if (dirichlet && i == 1) *ub = (T)u_b;
        factors(i, f_i, f_b, f_g);
        xg[dir] = ib + sgn * i;
        xi[dir] = ib - sgn * i;
        const double u_i = (double)*P.at(dir, 0, xi);
        *P.at(dir, 0, xg) = (T)(dirichlet ? f_i * u_i + f_b * u_b : f_i * u_i + f_b * u_b + f_g * cg);
        return;
    }
    T vb = dirichlet ? (T)(cg / ca) : *ub;
    constexpr int L = 4;  // layers loaded before any of them is stored
    for (int i0 = 1; i0 <= P.gcw; i0 += L)
    {
        double u_g[L], u_i[L];
#pragma unroll
        for (int k = 0; k < L; ++k)
            if (i0 + k <= P.gcw)
            {
                xg[dir] = ib + sgn * (i0 + k);
                xi[dir] = ib - sgn * (i0 + k);
                u_g[k] = (double)*P.at(dir, 0, xg);
                u_i[k] = (double)*P.at(dir, 0, xi);
            }
#pragma unroll
        for (int k = 0; k < L; ++k)
            if (i0 + k <= P.gcw)
            {
                factors(i0 + k, f_i, f_b, f_g);
                xi[dir] = ib - sgn * (i0 + k);
                *P.at(dir, 0, xi) = (T)(u_i[k] + f_i * u_g[k]);
                vb = (T)((double)vb + f_b * u_g[k]);
            }
    }
    *ub = vb;
}

__host__ __device__ inline void bd_edge(int loc, int* e, int* n1, int* n2, int* up1, int* up2)
{
    if (loc < 4)
    {
        *e = 0, *n1 = 1, *n2 = 2, *up1 = loc & 1, *up2 = (loc >> 1) & 1;
    }
    else if (loc < 8)
    {
        *e = 1, *n1 = 0, *n2 = 2, *up1 = (loc - 4) >> 1, *up2 = (loc - 4) & 1;
    }
    else
    {
        *e = 2, *n1 = 0, *n2 = 1, *up1 = (loc - 8) & 1, *up2 = (loc - 8) >> 1;
    }
}

// layers from an edge or corner box's normal face b inward to the mirror image of
// its outermost layer: the box's extent, more if it does not touch the patch
__host__ __device__ inline int bd_inward(int up, int b, int lo, int hi) { return up ? hi - b : b - lo; }

// cell data, 3-D edges.  Forward: work item = ghost value (all read values lie
// outside the edge box).  Adjoint: work item = possible target at one edge index: a
// value of the square from (b1, b2) inward to the mirror image (targets m, and on its
// sides those of the subtractions), a ghost value beside face 1 or beside face 2; it
// walks the sources in the reference's order (c2, then c1) and takes the updates that
// name it (none in the gap that a box off the patch leaves in the square).
template <typename T>
__device__ void bd_cc_edge(const BPatch<T>& P, int comp, int loc, const int* flo, const int* fhi, int adjoint, long t)
{
    int e, n1, n2, u1, u2;
    bd_edge(loc, &e, &n1, &n2, &u1, &u2);
    const int b1 = u1 ? P.ihi[n1] : P.ilo[n1], b2 = u2 ? P.ihi[n2] : P.ilo[n2];
    const int s1 = u1 ? 1 : -1, s2 = u2 ? 1 : -1;
    const int ne = fhi[e] - flo[e] + 1, k1 = fhi[n1] - flo[n1] + 1, k2 = fhi[n2] - flo[n2] + 1;
    const int ce = flo[e] + (int)(t % ne);
    const int r = (int)(t / ne);
    int x[3];
    x[e] = ce;
    auto val = [&](int i1, int i2) {
        x[n1] = i1, x[n2] = i2;
        return P.at(0, comp, x);
    };
    auto mir1 = [&](int c1) { return b1 + (b1 - c1 + s1); };
    auto mir2 = [&](int c2) { return b2 + (b2 - c2 + s2); };
    if (!adjoint)
    {
        const int c1 = flo[n1] + r % k1, c2 = flo[n2] + r / k1, m1 = mir1(c1), m2 = mir2(c2);
        const double v = (double)*val(m1, m2) + ((double)*val(b1, c2) - (double)*val(b1, m2)) +
                         ((double)*val(c1, b2) - (double)*val(m1, b2));
        *val(c1, c2) = (T)v;
        return;
    }
    const int q1 = bd_inward(u1, b1, flo[n1], fhi[n1]), q2 = bd_inward(u2, b2, flo[n2], fhi[n2]);
    int t1, t2;  // the target
    if (r < q1 * q2)
        t1 = b1 - s1 * (r % q1), t2 = b2 - s2 * (r / q1);
    else if (r < q1 * q2 + k1)
        t1 = flo[n1] + (r - q1 * q2), t2 = b2;
    else
        t1 = b1, t2 = flo[n2] + (r - q1 * q2 - k1);
    T v = *val(t1, t2);
    for (int c2 = flo[n2]; c2 <= fhi[n2]; ++c2)
        for (int c1 = flo[n1]; c1 <= fhi[n1]; ++c1)
        {
            const int m1 = mir1(c1), m2 = mir2(c2);
            const double Ug = (double)*val(c1, c2);
            if (t1 == m1 && t2 == m2) v = (T)((double)v + Ug);
            if (t1 == b1 && t2 == c2) v = (T)((double)v + Ug);
            if (t1 == c1 && t2 == b2) v = (T)((double)v + Ug);
            if (t1 == b1 && t2 == m2) v = (T)((double)v - Ug);
            if (t1 == m1 && t2 == b2) v = (T)((double)v - Ug);
        }
    *val(t1, t2) = v;
}

// cell data, corners (codim == ndim): as the edges, the sources in (z, y, x) order;
// targets: the cube from b inward to the mirror image, and the ghost values along
// axis d beside the corner cell
template <typename T>
__device__ void bd_cc_corner(const BPatch<T>& P, int comp, int loc, const int* flo, const int* fhi, int adjoint, long t)
{
    const int nd = P.ndim;
    int b[3] = {0, 0, 0}, s[3] = {0, 0, 0}, lo[3] = {0, 0, 0}, n[3] = {1, 1, 1};
    for (int d = 0; d < nd; ++d)
    {
        const int up = (loc >> d) & 1;
        b[d] = up ? P.ihi[d] : P.ilo[d];
        s[d] = up ? 1 : -1;
        lo[d] = flo[d];
        n[d] = fhi[d] - flo[d] + 1;
    }
    auto in = [&](int d) { return bd_inward(s[d] > 0, b[d], flo[d], fhi[d]); };
    const int cube = in(0) * in(1) * (nd == 3 ? in(2) : 1);
    auto source = [&](int q, int* x, int* m) {
        x[0] = lo[0] + q % n[0], x[1] = lo[1] + (q / n[0]) % n[1], x[2] = lo[2] + q / (n[0] * n[1]);
        m[2] = 0;
        for (int d = 0; d < nd; ++d) m[d] = b[d] + (b[d] - x[d] + s[d]);
    };
    auto on_axis = [&](const int* y, int d, int v) {  // y = b except y[d] = v
        bool same = y[d] == v;
        for (int o = 0; o < nd; ++o) same = same && (o == d || y[o] == b[o]);
        return same;
    };
    int x[3], m[3];
    if (!adjoint)
    {
        source((int)t, x, m);
        double v = (double)*P.at(0, comp, m);
        for (int d = 0; d < nd; ++d)
        {
            int pk[3] = {b[0], b[1], b[2]}, mk[3] = {b[0], b[1], b[2]};
            pk[d] = x[d];
            mk[d] = m[d];
            v = v + ((double)*P.at(0, comp, pk) - (double)*P.at(0, comp, mk));
        }
        *P.at(0, comp, x) = (T)v;
        return;
    }
    int y[3] = {b[0], b[1], b[2]};
    if (t < cube)
    {
        int r = (int)t;
        for (int d = 0; d < nd; ++d)
        {
            y[d] = b[d] - s[d] * (r % in(d));
            r /= in(d);
        }
    }
    else
    {
        int r = (int)t - cube, d = 0;
        while (d < nd - 1 && r >= n[d]) r -= n[d++];
        y[d] = lo[d] + r;
    }
    T* target = P.at(0, comp, y);
    T v = *target;
    for (int q = 0; q < n[0] * n[1] * n[2]; ++q)
    {
        source(q, x, m);
        const double Ug = (double)*P.at(0, comp, x);
        bool at_m = true;
        for (int d = 0; d < nd; ++d) at_m = at_m && y[d] == m[d];
        if (at_m) v = (T)((double)v + Ug);
        for (int d = 0; d < nd; ++d)
            if (on_axis(y, d, x[d])) v = (T)((double)v + Ug);
        for (int d = 0; d < nd; ++d)
            if (on_axis(y, d, m[d])) v = (T)((double)v - Ug);
    }
    *target = v;
}

// side data, 3-D edges, component comp extrapolated along the other normal axis.
// Adjoint: work item = (edge index, comp index), whose two targets collect from
// every layer; forward: (edge index, comp index, layer)
template <typename T>
__device__ void bd_sc_edge(const BPatch<T>& P, int comp, int loc, const int* flo, const int* fhi, int adjoint, long t)
{
    int e, n1, n2, u1, u2;
    bd_edge(loc, &e, &n1, &n2, &u1, &u2);
    const int other = comp == n1 ? n2 : n1;
    const int up = comp == n1 ? u2 : u1;
    const int bd = up ? P.ihi[other] : P.ilo[other], sh = up ? -1 : 1;
    const int ne = fhi[e] - flo[e] + 1, nc = fhi[comp] + 1 - flo[comp] + 1;
    const int c = (int)(t % ((long)ne * nc));
    int x[3];
    x[e] = flo[e] + c % ne;
    x[comp] = flo[comp] + c / ne;
    if (!(x[comp] < P.ilo[comp] || x[comp] > P.ihi[comp] + 1)) return;
    auto val = [&](int o) {
        x[other] = o;
        return P.at(comp, 0, x);
    };
    if (!adjoint)
    {
        const int o = flo[other] + (int)(t / ((long)ne * nc));
        const double del = (double)abs(o - bd);
        *val(o) = (T)((1.0 + del) * (double)*val(bd) - del * (double)*val(bd + sh));
        return;
    }
    T vb = *val(bd), vs = *val(bd + sh);
    for (int o = flo[other]; o <= fhi[other]; ++o)
    {
        const double del = (double)abs(o - bd), u_g = (double)*val(o);
        vb = (T)((double)vb + (1.0 + del) * u_g);
        vs = (T)((double)vs - del * u_g);
    }
    *val(bd) = vb;
    *val(bd + sh) = vs;
}

// side data, corners, one component.  Adjoint: work item = index along the
// component, whose targets (the corner's face value and one beside it per other
// axis) collect from every ghost value there; forward: ghost value
template <typename T>
__device__ void bd_sc_corner(const BPatch<T>& P, int comp, int loc, const int* flo, const int* fhi, int adjoint, long t)
{
    const int nd = P.ndim;
    int bd[3] = {0, 0, 0}, sh[3] = {0, 0, 0}, lo[3] = {0, 0, 0}, n[3] = {1, 1, 1};
    for (int d = 0; d < nd; ++d)
    {
        const int up = (loc >> d) & 1;
        bd[d] = up ? P.ihi[d] : P.ilo[d];
        sh[d] = up ? -1 : 1;
        lo[d] = flo[d];
        n[d] = fhi[d] - flo[d] + 1 + (d == comp ? 1 : 0);
    }
    int x[3], xb[3];
    auto weights = [&](double& dsum, double* del) {
        dsum = 1.0;
        for (int o = 0; o < nd; ++o)
            if (o != comp)
            {
                del[o] = (double)abs(x[o] - bd[o]);
                dsum = dsum + del[o];
            }
    };
    double dsum, del[3] = {0.0, 0.0, 0.0};
    if (!adjoint)
    {
        const int q = (int)t;
        x[0] = lo[0] + q % n[0], x[1] = lo[1] + (q / n[0]) % n[1], x[2] = lo[2] + q / (n[0] * n[1]);
        if (!(x[comp] < P.ilo[comp] || x[comp] > P.ihi[comp] + 1)) return;
        weights(dsum, del);
        for (int o = 0; o < 3; ++o) xb[o] = o < nd && o != comp ? bd[o] : x[o];
        double v = dsum * (double)*P.at(comp, 0, xb);
        for (int o = 0; o < nd; ++o)
            if (o != comp)
            {
                int xs[3] = {xb[0], xb[1], xb[2]};
                xs[o] += sh[o];
                v = v - del[o] * (double)*P.at(comp, 0, xs);
            }
        *P.at(comp, 0, x) = (T)v;
        return;
    }
    const int xc = lo[comp] + (int)t;
    if (!(xc < P.ilo[comp] || xc > P.ihi[comp] + 1)) return;
    for (int o = 0; o < 3; ++o) xb[o] = o == comp ? xc : bd[o];
    T* tb = P.at(comp, 0, xb);
    T vb = *tb, vs[3];
    T* ts[3] = {nullptr, nullptr, nullptr};
    for (int o = 0; o < nd; ++o)
        if (o != comp)
        {
            int xs[3] = {xb[0], xb[1], xb[2]};
            xs[o] += sh[o];
            ts[o] = P.at(comp, 0, xs);
            vs[o] = *ts[o];
        }
    const int n0 = comp == 0 ? 1 : n[0], n1 = comp == 1 ? 1 : n[1], n2 = comp == 2 ? 1 : n[2];
    for (int q = 0; q < n0 * n1 * n2; ++q)  // (z, y, x) order
    {
        x[0] = lo[0] + q % n0, x[1] = lo[1] + (q / n0) % n1, x[2] = lo[2] + q / (n0 * n1);
        x[comp] = xc;
        weights(dsum, del);
        const double u_g = (double)*P.at(comp, 0, x);
        vb = (T)((double)vb + dsum * u_g);
        for (int o = 0; o < nd; ++o)
            if (o != comp) vs[o] = (T)((double)vs[o] - del[o] * u_g);
    }
    *tb = vb;
    for (int o = 0; o < nd; ++o)
        if (o != comp) *ts[o] = vs[o];
}

constexpr int BDRY_B = 256;

template <typename T>
__global__ __launch_bounds__(BDRY_B) void k_phys_bdry(BdryArgs<T> a)
{
    const int2 blk = a.blocks[blockIdx.x];
    const BdryOp op = a.ops[blk.x];
    const long t = (long)blk.y + threadIdx.x;
    if (t >= op.count) return;
    const PatchDev& Q = a.patches[op.patch];
    BPatch<T> P;
    P.ndim = a.ndim;
    P.side = a.side;
    P.gcw = a.gcw;
    long vol = 1;
    for (int d = 0; d < 3; ++d)
    {
        P.ilo[d] = d < a.ndim ? Q.ilo[d] : 0;
        P.ihi[d] = d < a.ndim ? Q.ihi[d] : 0;
        if (d < a.ndim) vol *= (long)(Q.ihi[d] - Q.ilo[d] + 1 + 2 * a.gcw);
    }
    P.vol = vol;
    for (int d = 0; d < 3; ++d) P.arr[d] = d < a.narr ? a.arrays[op.patch * a.narr + d] : nullptr;
    const int* bx = a.boxes + 8 * op.box;
    const int loc = bx[1];
    const int lo[3] = {bx[2], bx[3], bx[4]}, hi[3] = {bx[5], bx[6], bx[7]};
    const int c = op.comp;
    // coefficient arrays per box: one per axis (side data) or per component (cell data)
    const long co = (long)op.box * (a.side ? a.ndim : a.depth) + c;
    switch (op.kind)
    {
    case B_CC_FACE:
        if (a.side)
        {
            int bhi[3] = {hi[0], hi[1], hi[2]};
            bhi[c] += 1;  // transverse component c: one more face along c
            bd_cc_face(P, c, 0, loc, P.ihi[loc / 2], lo, bhi, a.coef + a.coef_off[co], a.adjoint, a.dx, t);
        }
        else
            bd_cc_face(P, 0, c, loc, P.ihi[loc / 2], lo, hi, a.coef + a.coef_off[co], a.adjoint, a.dx, t);
        break;
    case B_SC_FACE: bd_sc_face(P, loc, lo, hi, a.coef + a.coef_off[co], a.adjoint, a.dx, t); break;
    case B_CC_EDGE: bd_cc_edge(P, c, loc, lo, hi, a.adjoint, t); break;
    case B_CC_CORNER: bd_cc_corner(P, c, loc, lo, hi, a.adjoint, t); break;
    case B_SC_EDGE: bd_sc_edge(P, c, loc, lo, hi, a.adjoint, t); break;
    case B_SC_CORNER: bd_sc_corner(P, c, loc, lo, hi, a.adjoint, t); break;
    }
}

// Index region (every value read or written) and work items of an operator.
struct BdryRegion
{
    long lo[3], hi[3];
};
BdryRegion bdry_region(const ibamr_plan* P, const BdryOp& op, const int* bx, bool adjoint, long* count)
{
    const PatchDev& Q = P->patches_h[op.patch];
    const int nd = P->ndim, loc = bx[1], g = P->data_gcw[0];
    const bool side = P->centering == IBAMR_SIDE;
    BdryRegion R{};
    long n[3] = {1, 1, 1};  // the box's extents, one more along the component of side data
    for (int d = 0; d < nd; ++d)
    {
        const int more = side && d == op.comp && op.kind != B_SC_FACE ? 1 : 0;
        R.lo[d] = bx[2 + d];
        R.hi[d] = bx[5 + d] + more;
        n[d] = R.hi[d] - R.lo[d] + 1;
    }
    auto layers = [&](int d, int up) -> long {
        return bd_inward(up, up ? Q.ihi[d] : Q.ilo[d], bx[2 + d], bx[5 + d]);
    };
    // along a normal axis d of an edge or corner: the box, and its mirror image inside
    // (cell data) or the two values that extrapolate (side data)
    auto inward = [&](int d, int up) {
        if (!side)
        {
            const long a = R.lo[d], b = R.hi[d];
            if (up)
                R.lo[d] = std::min(a, 2L * Q.ihi[d] - b + 1);
            else
                R.hi[d] = std::max(b, 2L * Q.ilo[d] - a - 1);
        }
        else if (d != op.comp)
        {
            if (up)
                R.lo[d] = std::min(R.lo[d], (long)Q.ihi[d] - 1);
            else
                R.hi[d] = std::max(R.hi[d], (long)Q.ilo[d] + 1);
        }
    };
    switch (op.kind)
    {
    case B_CC_FACE:
    {
        const int dir = loc / 2;
        R.lo[dir] = loc % 2 ? Q.ihi[dir] - g + 1 : Q.ilo[dir] - g;
        R.hi[dir] = loc % 2 ? Q.ihi[dir] + g : Q.ilo[dir] + g - 1;
        long c = g;
        for (int d = 0; d < nd; ++d)
            if (d != dir) c *= n[d];
        *count = c;
        break;
    }
    case B_SC_FACE:
    {
        const int dir = loc / 2, ib = loc % 2 ? Q.ihi[dir] + 1 : Q.ilo[dir];
        R.lo[dir] = ib - g;
        R.hi[dir] = ib + g;
        long c = adjoint ? 1 : g;
        for (int d = 0; d < nd; ++d)
            if (d != dir) c *= n[d];
        *count = c;
        break;
    }
    case B_CC_EDGE:
    case B_SC_EDGE:
    {
        int e, n1, n2, u1, u2;
        bd_edge(loc, &e, &n1, &n2, &u1, &u2);
        if (op.kind == B_CC_EDGE)
            *count = n[e] * (adjoint ? layers(n1, u1) * layers(n2, u2) + n[n1] + n[n2] : n[n1] * n[n2]);
        else
            *count = n[e] * n[op.comp] * (adjoint ? 1 : n[op.comp == n1 ? n2 : n1]);
        inward(n1, u1);
        inward(n2, u2);
        break;
    }
    case B_CC_CORNER:
    case B_SC_CORNER:
        if (op.kind == B_CC_CORNER && adjoint)
        {
            *count = 1;
            for (int d = 0; d < nd; ++d) *count *= layers(d, (loc >> d) & 1);
            for (int d = 0; d < nd; ++d) *count += n[d];
        }
        else if (op.kind == B_CC_CORNER)
            *count = n[0] * n[1] * n[2];
        else
            *count = adjoint ? n[op.comp] : n[0] * n[1] * n[2];
        for (int d = 0; d < nd; ++d) inward(d, (loc >> d) & 1);
        break;
    }
    return R;
}

// The operators of every patch in the reference's order (adjoint: corners, edges,
// codim-1 transverse, codim-1 normal; forward the reverse; boxes in the given order),
// each put into the first stage after every earlier operator of its patch and
// component whose region meets its own.
std::vector<std::vector<BdryOp>> bdry_stages(const ibamr_plan* P, const std::vector<int4>& patches,
                                             const std::vector<int>& boxes, bool adjoint)
{
    std::vector<std::vector<BdryOp>> stages;
    const int nd = P->ndim;
    const bool side = P->centering == IBAMR_SIDE;
    const int phases_adj[4] = {3, 2, 10, 11}, phases_fwd[4] = {11, 10, 2, 3};
    struct Done
    {
        int stage;
        BdryRegion r;
    };
    for (const int4& pl : patches)
    {
        std::vector<std::vector<Done>> done(side ? nd : P->depth);  // per component
        auto put = [&](int box, int kind, int comp) {
            BdryOp op{pl.x, box, kind, comp, 0};
            const BdryRegion r = bdry_region(P, op, &boxes[8 * (size_t)box], adjoint, &op.count);
            int st = 0;
            for (const Done& o : done[comp])
            {
                bool meet = true;
                for (int d = 0; d < nd; ++d) meet = meet && r.lo[d] <= o.r.hi[d] && o.r.lo[d] <= r.hi[d];
                if (meet) st = std::max(st, o.stage + 1);
            }
            done[comp].push_back(Done{st, r});
            if ((int)stages.size() <= st) stages.resize(st + 1);
            if (op.count > 0) stages[st].push_back(op);
        };
        for (int ph = 0; ph < 4; ++ph)
        {
            const int phase = adjoint ? phases_adj[ph] : phases_fwd[ph];
            for (int k = pl.y; k < pl.y + pl.z; ++k)
            {
                const int codim = boxes[8 * (size_t)k], loc = boxes[8 * (size_t)k + 1], dir = loc / 2;
                const int ncomp = side ? nd : P->depth;
                if ((phase == 3 && codim == 3) || (phase == 2 && codim == 2 && nd == 2))
                    for (int c = 0; c < ncomp; ++c) put(k, side ? B_SC_CORNER : B_CC_CORNER, c);
                else if (phase == 2 && codim == 2)
                {
                    if (!side)
                        for (int c = 0; c < ncomp; ++c) put(k, B_CC_EDGE, c);
                    else
                    {
                        int e, n1, n2, u1, u2;
                        bd_edge(loc, &e, &n1, &n2, &u1, &u2);
                        put(k, B_SC_EDGE, n1);
                        put(k, B_SC_EDGE, n2);
                    }
                }
                else if (phase == 10 && codim == 1)
                {
                    for (int c = 0; c < ncomp; ++c)
                        if (!side || c != dir) put(k, B_CC_FACE, c);
                }
                else if (phase == 11 && codim == 1 && side)
                    put(k, B_SC_FACE, dir);
            }
        }
    }
    return stages;
}
} // namespace
// Segments of the same-level ghost fill: the slabs of every patch array's ghost
// shell (see k_fill_level), FILL_SEG values each.
std::vector<int4> fill_segments(const ibamr_plan* P)
{
    std::vector<int4> segs;
    for (int i = 0; i < P->npatches; ++i)
    {
        const PatchDev& pd = P->patches_h[i];
        for (int c = 0; c < P->narr; ++c)
        {
            const int axis = P->centering == IBAMR_SIDE ? c : -1;
            for (int d = 0; d < P->ndim; ++d)
            {
                long m = P->data_gcw[d];
                for (int e = 0; e < P->ndim; ++e)
                    if (e != d)
                        m *= pd.ihi[e] - pd.ilo[e] + 1 + (e == axis ? 1 : 0) + (e < d ? 2 * P->data_gcw[e] : 0);
                for (int u = 0; u < 2; ++u)
                    for (long st = 0; st < m; st += FILL_SEG) segs.push_back(make_int4(i, c, 2 * d + u, (int)st));
            }
        }
    }
    return segs;
}
} // namespace ibamr

extern "C" {

int ibamr_plan_fill_periodic_ghosts(ibamr_plan* P, int slot, void* stream)
{
    if (!P) return fail(IBAMR_ERR_INVALID, "null plan");
    if (slot < 0 || slot >= MAX_SLOTS || !P->arrays_d[slot]) return fail(IBAMR_ERR_INVALID, "slot not bound");
    if (P->npatches != 1) return fail(IBAMR_ERR_INVALID, "periodic ghost fill needs a single-patch level");
    const PatchDev& pd = P->patches_h[0];
    for (int d = 0; d < P->ndim; ++d)
    {
        if (P->pshift[d] != pd.ihi[d] - pd.ilo[d] + 1 || pd.ilo[d] != P->dom_lo[d])
            return fail(IBAMR_ERR_INVALID, "periodic ghost fill needs a fully periodic domain covered by the patch");
    }
    // host copy of the pointer table: no device-to-host copy, so this can be captured
    const std::vector<void*>& ptrs = P->arrays_h[slot];
    hipStream_t s = static_cast<hipStream_t>(stream);
    PeriodicArgs q{};
    q.ncomps = P->centering == IBAMR_SIDE ? 1 : P->depth;
    long most = 0;
    for (int d = 0; d < 3; ++d)
    {
        q.g[d] = d < P->ndim ? P->data_gcw[d] : 0;
        q.N[d] = d < P->ndim ? pd.ihi[d] - pd.ilo[d] + 1 : 1;
    }
    for (int a = 0; a < P->narr; ++a)
    {
        const int axis = P->centering == IBAMR_SIDE ? a : -1;
        // the core along a side axis is the N faces [g, g+N): face N is the image of face 0
        for (int d = 0; d < 3; ++d) q.n[a][d] = q.N[d] + 2 * q.g[d] + (d == axis ? 1 : 0);
        const int* n = q.n[a];
        q.arr[a] = ptrs[a];
        q.sz[a] = (long)(n[2] - q.N[2]) * n[0] * n[1];
        q.sy[a] = (long)q.N[2] * (n[1] - q.N[1]) * n[0];
        q.sx[a] = (long)q.N[2] * q.N[1] * (n[0] - q.N[0]);
        most = std::max(most, q.sz[a] + q.sy[a] + q.sx[a]);
    }
    if (most == 0) return IBAMR_OK;
    const int B = 256;
    const dim3 G((unsigned)((most + B - 1) / B), (unsigned)(P->narr * q.ncomps));
    auto go = [&](auto tag) {
        using T = decltype(tag);
        if (most + B < (1L << 32))  // 32-bit shell indices (their divisions are several times cheaper)
            hipLaunchKernelGGL((k_fill_periodic<T, unsigned>), G, dim3(B), 0, s, q);
        else
            hipLaunchKernelGGL((k_fill_periodic<T, long>), G, dim3(B), 0, s, q);
    };
    if (P->precision == IBAMR_FP64)
        go((double)0);
    else
        go((float)0);
    HIP_OK(hipGetLastError());
    return IBAMR_OK;
}

int ibamr_plan_fill_ghosts(ibamr_plan* P, int slot, void* stream)
{
    if (!P) return fail(IBAMR_ERR_INVALID, "null plan");
    if (slot < 0 || slot >= MAX_SLOTS || !P->arrays_d[slot]) return fail(IBAMR_ERR_INVALID, "slot not bound");
    if (P->nfill_segs == 0) return IBAMR_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto go = [&](auto tag) -> int {
        using T = decltype(tag);
        FillArgs<T> a{};
        a.segs = P->fill_segs_d;
        a.patches = P->patches_d;
        a.arrays = reinterpret_cast<T* const*>(P->arrays_d[slot]);
        a.bin_patch_start = P->bin_patch_start_d;
        a.bin_patches = P->bin_patches_d;
        a.narr = P->narr;
        a.side = P->centering == IBAMR_SIDE;
        a.depth = P->depth;
        for (int d = 0; d < 3; ++d)
        {
            a.gcw[d] = P->data_gcw[d];
            a.dom_lo[d] = P->dom_lo[d];
            a.dom_hi[d] = P->dom_hi[d];
            a.pshift[d] = P->pshift[d];
            a.nb[d] = P->nb[d];
            a.nsb[d] = P->nsb[d];
        }
        a.bin = P->bin;
        if (P->ndim == 3)
            hipLaunchKernelGGL((k_fill_level<3, T>), dim3((unsigned)P->nfill_segs), dim3(256), 0, s, a);
        else
            hipLaunchKernelGGL((k_fill_level<2, T>), dim3((unsigned)P->nfill_segs), dim3(256), 0, s, a);
        HIP_OK(hipGetLastError());
        return IBAMR_OK;
    };
    return P->precision == IBAMR_FP64 ? go((double)0) : go((float)0);
}

// Coefficient values of a codim-1 box for array j: its tangential cells, one more
// along j for a side array tangential to the box (the coefficient box's
// tangential extension, CartSideRobinPhysBdryOp.cpp:913).
static long bdry_ncoef(const ibamr_plan* P, const ibamr_bdry_box& b, int j)
{
    const int dir = b.location / 2;
    long m = 1;
    for (int d = 0; d < P->ndim; ++d)
        if (d != dir) m *= (long)(b.upper[d] - b.lower[d] + 1 + (P->centering == IBAMR_SIDE && d == j ? 1 : 0));
    return m;
}

// Boxes with uniform coefficients (abg: [nboxes][arrays][3]) or coefficients over
// each codim-1 box (coefs: per codim-1 box in the given order and per array, a, b
// and g over the box's columns); exactly one of abg and coefs is given.
static int set_physical_boundary(ibamr_plan* P, const ibamr_bdry_box* boxes, int nboxes, const double* abg,
                                 const double* coefs, long ncoefs, bool varying)
{
    if (!P) return fail(IBAMR_ERR_INVALID, "null plan");
    if (nboxes < 0 || (nboxes > 0 && !boxes)) return fail(IBAMR_ERR_INVALID, "null boundary boxes");
    if (nboxes > 0 && !(varying ? (const void*)coefs : (const void*)abg))
        return fail(IBAMR_ERR_INVALID, "null boundary coefficients");
    for (int d = 1; d < P->ndim; ++d)
        if (P->data_gcw[d] != P->data_gcw[0])
            return fail(IBAMR_ERR_GHOST_WIDTH, "physical boundary operators need a uniform ghost width");
    if (P->centering == IBAMR_SIDE && P->depth != 1)
        return fail(IBAMR_ERR_INVALID, "physical boundary operators on side data of depth 1 only");
    const int g = P->data_gcw[0];
    // group by patch, keeping the given order inside each patch
    std::vector<std::vector<int>> per(P->npatches);
    for (int k = 0; k < nboxes; ++k)
    {
        const ibamr_bdry_box& b = boxes[k];
        if (b.patch < 0 || b.patch >= P->npatches)
            return fail(IBAMR_ERR_INVALID, "boundary box " + std::to_string(k) + ": bad patch index");
        if (b.codim < 1 || b.codim > P->ndim)
            return fail(IBAMR_ERR_INVALID, "boundary box " + std::to_string(k) + ": bad codimension");
        const int nloc = b.codim == 1 ? 2 * P->ndim : (b.codim == P->ndim ? (1 << P->ndim) : 12);
        if (b.location < 0 || b.location >= nloc)
            return fail(IBAMR_ERR_INVALID, "boundary box " + std::to_string(k) + ": bad location index");
        // every cell an operator touches must lie in the patch's ghost box
        const PatchDev& Q = P->patches_h[b.patch];
        for (int d = 0; d < P->ndim; ++d)
        {
            if (b.lower[d] > b.upper[d] || b.lower[d] < Q.ilo[d] - g || b.upper[d] > Q.ihi[d] + g)
                return fail(IBAMR_ERR_INVALID, "boundary box " + std::to_string(k) + " is not inside the ghost box");
        }
        if (b.codim == 1)
        {
            const int dir = b.location / 2;
            const int want = (b.location % 2) ? Q.ihi[dir] + 1 : Q.ilo[dir] - 1;
            if (b.lower[dir] != want || b.upper[dir] != want)
                return fail(IBAMR_ERR_INVALID, "boundary box " + std::to_string(k) + ": a codim-1 box is the cell "
                                               "layer just outside its face");
            for (int d = 0; d < P->ndim; ++d)
                if (d != dir && (b.lower[d] < Q.ilo[d] || b.upper[d] > Q.ihi[d]))
                    return fail(IBAMR_ERR_INVALID, "boundary box " + std::to_string(k) + ": a codim-1 box spans at "
                                                   "most its face");
        }
        else
        {
            // codim 2 / ndim: outside the patch, within the ghost width, on the sides the location names
            int up[3] = {-1, -1, -1};  // -1: along the box (edge direction)
            if (b.codim == P->ndim)
                for (int d = 0; d < P->ndim; ++d) up[d] = (b.location >> d) & 1;
            else
            {
                const int l = b.location;
                if (l < 4)
                    up[1] = l & 1, up[2] = (l >> 1) & 1;
                else if (l < 8)
                    up[0] = (l - 4) >> 1, up[2] = (l - 4) & 1;
                else
                    up[0] = (l - 8) & 1, up[1] = (l - 8) >> 1;
            }
            for (int d = 0; d < P->ndim; ++d)
            {
                if (up[d] < 0) continue;
                const bool ok = up[d] ? b.lower[d] > Q.ihi[d] : b.upper[d] < Q.ilo[d];
                if (!ok)
                    return fail(IBAMR_ERR_INVALID, "boundary box " + std::to_string(k) +
                                                       ": an edge or corner box lies outside the patch on its sides");
            }
        }
        per[b.patch].push_back(k);
    }
    const int narr = P->centering == IBAMR_SIDE ? P->ndim : P->depth;
    // where box k's coefficients for array j start in the caller's coefs
    std::vector<long> uoff((size_t)nboxes * narr, 0);
    long need = 0;
    for (int k = 0; k < nboxes; ++k)
        if (boxes[k].codim == 1)
            for (int j = 0; j < narr; ++j)
            {
                uoff[(size_t)k * narr + j] = need;
                need += 3 * bdry_ncoef(P, boxes[k], j);
            }
    if (varying && ncoefs != need)
        return fail(IBAMR_ERR_INVALID, "boundary coefficients: " + std::to_string(ncoefs) + " values given, the boxes "
                                       "need " + std::to_string(need));
    std::vector<int4> pl;
    std::vector<int> bx;
    std::vector<double> cf;
    std::vector<long> cfo;
    for (int p = 0; p < P->npatches; ++p)
    {
        if (per[p].empty()) continue;
        pl.push_back(make_int4(p, (int)(bx.size() / 8), (int)per[p].size(), 0));
        for (int k : per[p])
        {
            const ibamr_bdry_box& b = boxes[k];
            const int v[8] = {b.codim, b.location, b.lower[0], b.lower[1], P->ndim == 3 ? b.lower[2] : 0,
                              b.upper[0], b.upper[1], P->ndim == 3 ? b.upper[2] : 0};
            bx.insert(bx.end(), v, v + 8);
            for (int j = 0; j < narr; ++j)
            {
                cfo.push_back((long)cf.size());
                if (b.codim != 1) continue;
                const long m = bdry_ncoef(P, b, j);
                if (varying)
                {
                    const double* u = coefs + uoff[(size_t)k * narr + j];
                    cf.insert(cf.end(), u, u + 3 * m);
                }
                else
                    for (int c = 0; c < 3; ++c) cf.insert(cf.end(), (size_t)m, abg[3 * ((long)k * narr + j) + c]);
            }
        }
    }
    dfree(P->bdry_mem_d);
    P->bdry_mem_d = nullptr;
    P->nbdry_patches = 0;
    if (pl.empty()) return IBAMR_OK;
    if (cf.empty()) cf.push_back(0.0);
    // one allocation for all tables
    std::vector<BdryOp> ops[2];
    std::vector<int2> blocks[2];
    for (int m = 0; m < 2; ++m)
    {
        P->bdry_stage_start[m].clear();
        for (const std::vector<BdryOp>& st : bdry_stages(P, pl, bx, m == 1))
        {
            P->bdry_stage_start[m].push_back((int)blocks[m].size());
            for (const BdryOp& op : st)
            {
                for (long t = 0; t < op.count; t += BDRY_B) blocks[m].push_back(make_int2((int)ops[m].size(), (int)t));
                ops[m].push_back(op);
            }
        }
        P->bdry_stage_start[m].push_back((int)blocks[m].size());
    }
    size_t bytes = 0;
    auto place = [&](size_t n) {
        const size_t at = bytes;
        bytes += (n + 15) / 16 * 16;
        return at;
    };
    const size_t at_coef = place(sizeof(double) * cf.size()), at_off = place(sizeof(long) * cfo.size());
    const size_t at_box = place(sizeof(int) * bx.size());
    const size_t at_ops[2] = {place(sizeof(BdryOp) * ops[0].size()), place(sizeof(BdryOp) * ops[1].size())};
    const size_t at_blocks[2] = {place(sizeof(int2) * blocks[0].size()), place(sizeof(int2) * blocks[1].size())};
    HIP_OK(hipMalloc(&P->bdry_mem_d, bytes));
    P->bdry_box_d = reinterpret_cast<int*>(P->bdry_mem_d + at_box);
    P->bdry_coef_d = reinterpret_cast<double*>(P->bdry_mem_d + at_coef);
    P->bdry_coef_off_d = reinterpret_cast<long*>(P->bdry_mem_d + at_off);
    // two copies (a caller whose coefficients change in time sets them every step):
    // the coefficients, and the other tables behind them
    std::vector<char> mem(bytes - at_off);
    auto put = [&](size_t at, const auto& v) {
        if (!v.empty()) std::memcpy(mem.data() + (at - at_off), v.data(), sizeof(v[0]) * v.size());
    };
    put(at_off, cfo);
    put(at_box, bx);
    for (int m = 0; m < 2; ++m)
    {
        P->bdry_ops_d[m] = reinterpret_cast<BdryOp*>(P->bdry_mem_d + at_ops[m]);
        P->bdry_blocks_d[m] = reinterpret_cast<int2*>(P->bdry_mem_d + at_blocks[m]);
        put(at_ops[m], ops[m]);
        put(at_blocks[m], blocks[m]);
    }
    HIP_OK(hipMemcpy(P->bdry_coef_d, cf.data(), sizeof(double) * cf.size(), hipMemcpyHostToDevice));
    HIP_OK(hipMemcpy(P->bdry_mem_d + at_off, mem.data(), mem.size(), hipMemcpyHostToDevice));
    P->nbdry_patches = (int)pl.size();
    return IBAMR_OK;
}

int ibamr_plan_set_physical_boundary(ibamr_plan* P, const ibamr_bdry_box* boxes, int nboxes, const double* abg)
{
    return set_physical_boundary(P, boxes, nboxes, abg, nullptr, 0, false);
}

int ibamr_plan_set_physical_boundary_coefs(ibamr_plan* P, const ibamr_bdry_box* boxes, int nboxes,
                                           const double* coefs, long ncoefs)
{
    return set_physical_boundary(P, boxes, nboxes, nullptr, coefs, ncoefs, true);
}

static int phys_bdry_launch(ibamr_plan* P, int slot, int adjoint, void* stream)
{
    if (!P) return fail(IBAMR_ERR_INVALID, "null plan");
    if (slot < 0 || slot >= MAX_SLOTS || !P->arrays_d[slot]) return fail(IBAMR_ERR_INVALID, "slot not bound");
    if (P->nbdry_patches == 0) return IBAMR_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    auto go = [&](auto tag) -> int {
        using T = decltype(tag);
        BdryArgs<T> a{};
        a.ops = P->bdry_ops_d[adjoint];
        a.boxes = P->bdry_box_d;
        a.coef = P->bdry_coef_d;
        a.coef_off = P->bdry_coef_off_d;
        a.patches = P->patches_d;
        a.arrays = reinterpret_cast<T* const*>(P->arrays_d[slot]);
        a.ndim = P->ndim;
        a.side = P->centering == IBAMR_SIDE;
        a.depth = P->depth;
        a.narr = P->narr;
        a.gcw = P->data_gcw[0];
        a.adjoint = adjoint;
        for (int d = 0; d < 3; ++d) a.dx[d] = P->dx[d];
        const std::vector<int>& start = P->bdry_stage_start[adjoint];
        for (size_t k = 0; k + 1 < start.size(); ++k)
        {
            if (start[k + 1] == start[k]) continue;
            a.blocks = P->bdry_blocks_d[adjoint] + start[k];
            hipLaunchKernelGGL(k_phys_bdry<T>, dim3((unsigned)(start[k + 1] - start[k])), dim3(BDRY_B), 0, s, a);
        }
        HIP_OK(hipGetLastError());
        return IBAMR_OK;
    };
    return P->precision == IBAMR_FP64 ? go((double)0) : go((float)0);
}

int ibamr_plan_accumulate_physical_boundary(ibamr_plan* P, int slot, void* stream)
{
    return phys_bdry_launch(P, slot, 1, stream);
}

int ibamr_plan_fill_physical_boundary(ibamr_plan* P, int slot, void* stream)
{
    return phys_bdry_launch(P, slot, 0, stream);
}

} // extern "C"
