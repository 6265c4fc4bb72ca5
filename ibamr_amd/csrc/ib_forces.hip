// ib_forces.hip -- Lagrangian force generation on the GPU: springs, beams
// (three-point bending) and target points, the forces IBStandardForceGen
// computes before the spread (src/IB/IBStandardForceGen.cpp:254-305; springs
// :814-930 with default_spring_force, include/ibamr/IBSpringForceFunctions.h:104,
// or another registered force function; beams :1038-1147; target points
// :1202-1299).
//
// The reference keeps a map force_fcn_idx -> function pointer
// (registerSpringForceFunction, :133-140) and resolves every spring's index to
// its function when the level's data is set up (:728-790).  Host function
// pointers cannot run on the GPU, so the map here holds built-in device laws
// (spring_tension below), resolved per spring the same way, when the spring
// parameters are set.
//
// The reference loops over springs, then beams, then target points, adding each
// element's force into its nodes in element order (a scatter into F_ghost,
// which starts at zero), and finally adds F_ghost to F.  Here one thread per node
// walks a node -> (element, role) list kept in exactly that order and evaluates
// each element's force with the reference's arithmetic where it adds it, so every
// node's force is the same sequence of floating-point operations as the reference
// loop: bitwise identical, and deterministic (no atomics).  An element is evaluated
// once per node it touches (2 or 3 times): its arithmetic costs less than writing
// its force and gathering it back.
#include "ibamr_amd.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <map>
#include <string>
#include <type_traits>
#include <vector>

namespace ibamr
{
int set_error(int code, const std::string& msg);
}

namespace
{
using ibamr::set_error;

enum Role : int
{
    R_SPRING_MASTER = 0,
    R_SPRING_SLAVE = 1,
    R_BEAM_MASTER = 2,
    R_BEAM_NEXT = 3,
    R_BEAM_PREV = 4,
    R_TARGET = 5
};

#define F_HIP(expr)                                                                               \
    do                                                                                            \
    {                                                                                             \
        hipError_t e_ = (expr);                                                                   \
        if (e_ != hipSuccess) return set_error(IBAMR_ERR_DEVICE, std::string(#expr ": ") + hipGetErrorString(e_)); \
    } while (0)

// Tension T(R) of spring law `law` with parameters p[0 .. np):
//   IBAMR_SPRING_HOOKEAN: p[0] (R - p[1]) (default_spring_force,
//     IBSpringForceFunctions.h:104-107);
//   IBAMR_SPRING_LINEAR_STRAIN: p[0] (R / p[1] - 1) (the linear_spring_force
//     examples/IB/explicit/ex3/example.cpp:58-63 registers);
//   IBAMR_SPRING_POLYNOMIAL: x (p[0] + x (p[2] + ... + x p[np-1])), x = R - p[1].
__device__ inline double spring_tension(int law, const double* __restrict__ p, int np, double R)
{
    if (law == IBAMR_SPRING_LINEAR_STRAIN) return p[0] * (R / p[1] - 1.0);
    if (law == IBAMR_SPRING_POLYNOMIAL)
    {
        const double x = R - p[1];
        double h = np > 2 ? p[np - 1] : p[0];
        for (int m = np - 2; m >= 2; --m) h = p[m] + x * h;
        if (np > 2) h = p[0] + x * h;
        return x * h;
    }
    return p[0] * (R - p[1]);
}

struct ForceArgs
{
    int n;
    const int* start;
    const int* ent;       // element << 3 | role, or pairs (role, element) when an element number needs more bits
    int packed;
    const int *s_m, *s_s;
    const int *s_law, *s_off;  // null: every spring Hookean with two parameters
    const double* s_par;
    const int *b_m, *b_n, *b_p;
    const double *b_K, *b_c;
    const double *t_K, *t_E, *t_X0;
};

// LANES lanes per node take its list that many entries at a time: each evaluates one
// entry, then all add the entries' forces in list order.  Nodes of few entries are
// bound by memory (per node of a ring with springs, beams and a target point at every
// 4th node about 220 bytes of lists, parameters, positions and force; 1.5 M nodes FP64:
// 85 us a call, 139 us as a spring, a beam and a gather kernel), nodes of many by the
// latency of the chain start -> entry -> element -> position.  1 / 2 / 8 lanes, us:
// springs of a ring (2 entries a node, 10^6 nodes) 19 / 18 / 51, beams (3) 30 / 30 / 63,
// spring networks of valence 12 and 26 (200 k nodes) 115 / 90 / 47 and 306 / 220 / 107
// (287 as a spring and a gather kernel).
template <int NDIM, typename TF, typename TU, int LANES>
__global__ __launch_bounds__(256) void k_node_forces(ForceArgs a, const double* __restrict__ X,
                                                     const TU* __restrict__ U, TF* __restrict__ F, int overwrite)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)a.n * LANES) return;
    const int v = (int)(t / LANES), l = threadIdx.x % LANES;
    double acc[NDIM], Xv[NDIM];
#pragma unroll
    for (int d = 0; d < NDIM; ++d)
    {
        acc[d] = 0.0;
        Xv[d] = X[(size_t)NDIM * v + d];
    }
    // add(d, f_d) with what entry e adds to the node's force; false: nothing (skipped)
    auto entry = [&](int e, auto add) {
        int role, k;
        if (a.packed)
        {
            const unsigned en = (unsigned)a.ent[e];
            role = (int)(en & 7u);
            k = (int)(en >> 3);
        }
        else
        {
            role = a.ent[2 * (size_t)e];
            k = a.ent[2 * (size_t)e + 1];
        }
        if (role <= R_SPRING_SLAVE)
        {
            // D = X_slave - X_master, R = |D|, T/R = T(R) / R, F = (T/R) D; skipped when
            // R < DBL_EPSILON (IBStandardForceGen.cpp:903-911)
            const bool master = role == R_SPRING_MASTER;
            const size_t o = (size_t)NDIM * (master ? a.s_s[k] : a.s_m[k]);
            double D[NDIM];
#pragma unroll
            for (int d = 0; d < NDIM; ++d)
            {
                const double Xo = X[o + d];
                D[d] = master ? Xo - Xv[d] : Xv[d] - Xo;
            }
            double R2 = D[0] * D[0] + D[1] * D[1];
            if (NDIM == 3) R2 = R2 + D[NDIM - 1] * D[NDIM - 1];
            const double R = sqrt(R2);
            if (R < DBL_EPSILON) return false;
            double T;
            if (a.s_law)
            {
                const int q = a.s_off[k];
                T = spring_tension(a.s_law[k], a.s_par + q, a.s_off[k + 1] - q, R);
            }
            else
                T = spring_tension(IBAMR_SPRING_HOOKEAN, a.s_par + 2 * (size_t)k, 2, R);
            const double T_over_R = T / R;
#pragma unroll
            for (int d = 0; d < NDIM; ++d)
            {
                const double q = T_over_R * D[d];
                add(d, master ? q : -q);
            }
        }
        else if (role <= R_BEAM_PREV)
        {
            // F = K (X_next + X_prev - 2 X_master - curvature) (IBStandardForceGen.cpp:1129-1131)
            const size_t im = (size_t)NDIM * (role == R_BEAM_MASTER ? v : a.b_m[k]),
                         in = (size_t)NDIM * (role == R_BEAM_NEXT ? v : a.b_n[k]),
                         ip = (size_t)NDIM * (role == R_BEAM_PREV ? v : a.b_p[k]);
            const double K = a.b_K[k];
#pragma unroll
            for (int d = 0; d < NDIM; ++d)
            {
                const double q = K * (((X[in + d] + X[ip + d]) - 2.0 * X[im + d]) - a.b_c[(size_t)NDIM * k + d]);
                add(d, role == R_BEAM_MASTER ? 2.0 * q : -q);
            }
        }
        else  // target point (IBStandardForceGen.cpp:1285-1288)
        {
            const double K = a.t_K[k], E = a.t_E[k];
#pragma unroll
            for (int d = 0; d < NDIM; ++d)
            {
                const double u = U ? (double)U[(size_t)NDIM * v + d] : 0.0;
                add(d, K * (a.t_X0[(size_t)NDIM * k + d] - Xv[d]) - E * u);
            }
        }
        return true;
    };
    const int e1 = a.start[v + 1];
    if constexpr (LANES == 1)
    {
        for (int e = a.start[v]; e < e1; ++e) entry(e, [&](int d, double f) { acc[d] = acc[d] + f; });
    }
    else
    {
        for (int e0 = a.start[v]; e0 < e1; e0 += LANES)
        {
            double f[NDIM] = {};
            const int some = e0 + l < e1 && entry(e0 + l, [&](int d, double g) { f[d] = g; }) ? 1 : 0;
            const int m = min(LANES, e1 - e0);
            for (int j = 0; j < m; ++j)
            {
                const int take = __shfl(some, j, LANES);
#pragma unroll
                for (int d = 0; d < NDIM; ++d)
                {
                    const double g = __shfl(f[d], j, LANES);
                    acc[d] = take ? acc[d] + g : acc[d];
                }
            }
        }
        if (l != 0) return;
    }
    // F += F_ghost (VecAXPY with alpha 1, :300), or F = F_ghost
#pragma unroll
    for (int d = 0; d < NDIM; ++d)
    {
        const size_t i = (size_t)NDIM * v + d;
        F[i] = overwrite ? (TF)acc[d] : (TF)((double)F[i] + acc[d]);
    }
}

__global__ void k_copy_positions(long n, const double* __restrict__ X, double* __restrict__ out)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = X[i];
}

template <typename T>
int dev_copy(T** dst, const T* src, size_t n)
{
    *dst = nullptr;
    if (n == 0) return IBAMR_OK;
    F_HIP(hipMalloc(dst, sizeof(T) * n));
    F_HIP(hipMemcpy(*dst, src, sizeof(T) * n, hipMemcpyHostToDevice));
    return IBAMR_OK;
}

void dfree(void* p)
{
    if (p) (void)hipFree(p);
}
} // namespace

struct ibamr_forces
{
    int ndim = 3, n = 0, ns = 0, nb = 0, nt = 0;
    int *s_m = nullptr, *s_s = nullptr;
    int *s_law = nullptr, *s_off = nullptr;  // per spring: law, first parameter ([ns + 1]); null: the default
                                             // force function for every spring, {kappa, rest} each
    double* s_par = nullptr;
    std::map<int, int> registry{{0, IBAMR_SPRING_HOOKEAN}};  // force function index -> law
    int *b_m = nullptr, *b_n = nullptr, *b_p = nullptr;
    double *b_K = nullptr, *b_c = nullptr;
    int* t_i = nullptr;
    double *t_K = nullptr, *t_E = nullptr, *t_X0 = nullptr;
    int* start = nullptr;
    int* ent = nullptr;
    double* Xc = nullptr;  // [n][ndim] positions while F is written over them
    bool packed = true;
    int lanes = 1;  // lanes per node of k_node_forces
};

extern "C" {

int ibamr_forces_destroy(ibamr_forces* f)
{
    if (!f) return IBAMR_OK;
    for (void* p : {(void*)f->s_m, (void*)f->s_s, (void*)f->s_law, (void*)f->s_off, (void*)f->s_par, (void*)f->b_m, (void*)f->b_n,
                    (void*)f->b_p, (void*)f->b_K, (void*)f->b_c, (void*)f->t_i, (void*)f->t_K, (void*)f->t_E,
                    (void*)f->t_X0, (void*)f->start, (void*)f->ent, (void*)f->Xc})
        dfree(p);
    delete f;
    return IBAMR_OK;
}

int ibamr_forces_create(ibamr_forces** out, int ndim, int npoints, int nsprings, const int* spring_master,
                        const int* spring_slave, const double* spring_kappa, const double* spring_rest, int nbeams,
                        const int* beam_master, const int* beam_next, const int* beam_prev,
                        const double* beam_rigidity, const double* beam_curvature, int ntargets,
                        const int* target_node, const double* target_kappa, const double* target_eta,
                        const double* target_X0)
{
    if (!out) return set_error(IBAMR_ERR_INVALID, "null argument");
    *out = nullptr;
    if (ndim != 2 && ndim != 3) return set_error(IBAMR_ERR_INVALID, "ndim must be 2 or 3");
    if (npoints < 0 || nsprings < 0 || nbeams < 0 || ntargets < 0) return set_error(IBAMR_ERR_INVALID, "negative count");
    if ((nsprings > 0 && (!spring_master || !spring_slave || !spring_kappa || !spring_rest)) ||
        (nbeams > 0 && (!beam_master || !beam_next || !beam_prev || !beam_rigidity || !beam_curvature)) ||
        (ntargets > 0 && (!target_node || !target_kappa || !target_eta || !target_X0)))
        return set_error(IBAMR_ERR_INVALID, "null element array");
    auto bad = [&](int i) { return i < 0 || i >= npoints; };
    // node -> (role, element) lists in the reference's order: springs, beams,
    // target points, each in element order
    std::vector<std::vector<int2>> lists((size_t)npoints);
    for (int k = 0; k < nsprings; ++k)
    {
        if (bad(spring_master[k]) || bad(spring_slave[k]) || spring_master[k] == spring_slave[k])
            return set_error(IBAMR_ERR_INVALID, "spring " + std::to_string(k) + ": bad node index");
        lists[spring_master[k]].push_back(make_int2(R_SPRING_MASTER, k));
        lists[spring_slave[k]].push_back(make_int2(R_SPRING_SLAVE, k));
    }
    for (int k = 0; k < nbeams; ++k)
    {
        if (bad(beam_master[k]) || bad(beam_next[k]) || bad(beam_prev[k]) || beam_master[k] == beam_next[k] ||
            beam_master[k] == beam_prev[k])
            return set_error(IBAMR_ERR_INVALID, "beam " + std::to_string(k) + ": bad node index");
        lists[beam_master[k]].push_back(make_int2(R_BEAM_MASTER, k));
        lists[beam_next[k]].push_back(make_int2(R_BEAM_NEXT, k));
        lists[beam_prev[k]].push_back(make_int2(R_BEAM_PREV, k));
    }
    for (int k = 0; k < ntargets; ++k)
    {
        if (bad(target_node[k])) return set_error(IBAMR_ERR_INVALID, "target point " + std::to_string(k) + ": bad node index");
        lists[target_node[k]].push_back(make_int2(R_TARGET, k));
    }
    // an entry is one int (element << 3 | role) while the element numbers fit
    const bool packed = std::max(nsprings, std::max(nbeams, ntargets)) <= (1 << 29);
    std::vector<int> start((size_t)npoints + 1, 0);
    std::vector<int> ent;
    size_t nent = 0;
    for (int v = 0; v < npoints; ++v)
    {
        start[v] = (int)nent;
        for (const int2& q : lists[v])
        {
            if (packed)
                ent.push_back((int)((unsigned)q.y << 3 | (unsigned)q.x));
            else
            {
                ent.push_back(q.x);
                ent.push_back(q.y);
            }
        }
        nent += lists[v].size();
    }
    start[npoints] = (int)nent;

    ibamr_forces* f = new ibamr_forces();
    f->packed = packed;
    // 8 lanes per node for lists of 12 entries and more on average, or where one is so
    // long that it takes longer than all others (one hub of 1000 springs: 535 us with one
    // lane, 235 with 8; see k_node_forces)
    size_t longest = 0;
    for (const auto& l : lists) longest = std::max(longest, l.size());
    f->lanes = nent >= 12 * (size_t)npoints || longest >= 256 ? 8 : 1;
    f->ndim = ndim;
    f->n = npoints;
    f->ns = nsprings;
    f->nb = nbeams;
    f->nt = ntargets;
    int rc = IBAMR_OK;
    auto chk = [&](int r) {
        if (rc == IBAMR_OK) rc = r;
    };
    chk(dev_copy(&f->s_m, spring_master, (size_t)nsprings));
    chk(dev_copy(&f->s_s, spring_slave, (size_t)nsprings));
    {
        // the default force function: law IBAMR_SPRING_HOOKEAN with {kappa, rest}
        std::vector<double> par((size_t)nsprings * 2);
        for (int k = 0; k < nsprings; ++k)
        {
            par[2 * (size_t)k] = spring_kappa[k];
            par[2 * (size_t)k + 1] = spring_rest[k];
        }
        chk(dev_copy(&f->s_par, par.data(), par.size()));
    }
    chk(dev_copy(&f->b_m, beam_master, (size_t)nbeams));
    chk(dev_copy(&f->b_n, beam_next, (size_t)nbeams));
    chk(dev_copy(&f->b_p, beam_prev, (size_t)nbeams));
    chk(dev_copy(&f->b_K, beam_rigidity, (size_t)nbeams));
    chk(dev_copy(&f->b_c, beam_curvature, (size_t)nbeams * ndim));
    chk(dev_copy(&f->t_i, target_node, (size_t)ntargets));
    chk(dev_copy(&f->t_K, target_kappa, (size_t)ntargets));
    chk(dev_copy(&f->t_E, target_eta, (size_t)ntargets));
    chk(dev_copy(&f->t_X0, target_X0, (size_t)ntargets * ndim));
    chk(dev_copy(&f->start, start.data(), start.size()));
    chk(dev_copy(&f->ent, ent.data(), ent.size()));
    // here and not at its first use, which may be under capture
    if (rc == IBAMR_OK && nsprings + nbeams > 0 &&
        hipMalloc(&f->Xc, sizeof(double) * (size_t)npoints * ndim) != hipSuccess)
        rc = set_error(IBAMR_ERR_DEVICE, "hipMalloc of position scratch failed");
    if (rc != IBAMR_OK)
    {
        ibamr_forces_destroy(f);
        return rc;
    }
    *out = f;
    return IBAMR_OK;
}

int ibamr_forces_register_spring_function(ibamr_forces* f, int force_fcn_index, int law)
{
    if (!f) return set_error(IBAMR_ERR_INVALID, "null force object");
    if (law != IBAMR_SPRING_HOOKEAN && law != IBAMR_SPRING_LINEAR_STRAIN && law != IBAMR_SPRING_POLYNOMIAL)
        return set_error(IBAMR_ERR_INVALID, "unknown spring law " + std::to_string(law));
    f->registry[force_fcn_index] = law;
    return IBAMR_OK;
}

int ibamr_forces_set_spring_parameters(ibamr_forces* f, const int* force_fcn_idx, const int* param_offsets,
                                       const double* params)
{
    if (!f) return set_error(IBAMR_ERR_INVALID, "null force object");
    const int ns = f->ns;
    if (ns == 0) return IBAMR_OK;
    if (!force_fcn_idx || !param_offsets || (!params && param_offsets[ns] > 0))
        return set_error(IBAMR_ERR_INVALID, "null spring parameter array");
    if (param_offsets[0] != 0) return set_error(IBAMR_ERR_INVALID, "spring parameter offsets must start at 0");
    std::vector<int> law((size_t)ns);
    for (int k = 0; k < ns; ++k)
    {
        const auto it = f->registry.find(force_fcn_idx[k]);
        if (it == f->registry.end())
            return set_error(IBAMR_ERR_INVALID, "spring " + std::to_string(k) + ": no spring force function is "
                                                "registered under index " + std::to_string(force_fcn_idx[k]));
        const int np = param_offsets[k + 1] - param_offsets[k];
        if (np < 2)
            return set_error(IBAMR_ERR_INVALID, "spring " + std::to_string(k) + ": " + std::to_string(np) +
                                                    " parameters (at least stiffness and rest length)");
        law[k] = it->second;
    }
    int* d_law = nullptr;
    int* d_off = nullptr;
    double* d_par = nullptr;
    int rc = dev_copy(&d_law, law.data(), law.size());
    if (rc == IBAMR_OK) rc = dev_copy(&d_off, param_offsets, (size_t)ns + 1);
    if (rc == IBAMR_OK) rc = dev_copy(&d_par, params, (size_t)param_offsets[ns]);
    if (rc != IBAMR_OK)
    {
        dfree(d_law);
        dfree(d_off);
        dfree(d_par);
        return rc;
    }
    dfree(f->s_law);
    dfree(f->s_off);
    dfree(f->s_par);
    f->s_law = d_law;
    f->s_off = d_off;
    f->s_par = d_par;
    return IBAMR_OK;
}

int ibamr_forces_compute(ibamr_forces* f, void* F, int f_precision, const double* X, const void* U,
                         int u_precision, int mode, void* stream)
{
    if (!f) return set_error(IBAMR_ERR_INVALID, "null force object");
    if (f->n == 0) return IBAMR_OK;
    if (!F || !X) return set_error(IBAMR_ERR_INVALID, "null F or X");
    if (f_precision != IBAMR_FP64 && f_precision != IBAMR_FP32C) return set_error(IBAMR_ERR_INVALID, "bad precision");
    if (U && u_precision != IBAMR_FP64 && u_precision != IBAMR_FP32C)
        return set_error(IBAMR_ERR_INVALID, "bad velocity precision");
    if (mode != IBAMR_SPREAD_ACCUMULATE && mode != IBAMR_SPREAD_OVERWRITE) return set_error(IBAMR_ERR_INVALID, "bad mode");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int B = 256;
    const int ow = mode == IBAMR_SPREAD_OVERWRITE ? 1 : 0;
    // springs and beams read other nodes' positions: from a copy where F lies over X
    const size_t nv = (size_t)f->n * f->ndim;
    const char *f0 = static_cast<const char*>(F), *f1 = f0 + nv * (f_precision == IBAMR_FP64 ? 8 : 4);
    const char *x0 = reinterpret_cast<const char*>(X), *x1 = x0 + nv * 8;
    if (f->Xc && f0 < x1 && x0 < f1)
    {
        hipLaunchKernelGGL(k_copy_positions, dim3((unsigned)((nv + B - 1) / B)), dim3(B), 0, s, (long)nv, X, f->Xc);
        F_HIP(hipGetLastError());
        X = f->Xc;
    }
    const int lanes = f->lanes;
    const dim3 grid((unsigned)(((long)f->n * lanes + B - 1) / B));
    const ForceArgs a{f->n,   f->start, f->ent, f->packed ? 1 : 0, f->s_m, f->s_s, f->s_law, f->s_off, f->s_par, f->b_m,
                      f->b_n, f->b_p,   f->b_K, f->b_c,            f->t_K, f->t_E, f->t_X0};
    auto go = [&](auto dim, auto tf, auto tu) {
        using TF = decltype(tf);
        using TU = decltype(tu);
        constexpr int NDIM = decltype(dim)::value;
        const auto kernel = lanes == 8 ? k_node_forces<NDIM, TF, TU, 8> : k_node_forces<NDIM, TF, TU, 1>;
        hipLaunchKernelGGL(kernel, grid, dim3(B), 0, s, a, X, static_cast<const TU*>(U), static_cast<TF*>(F), ow);
    };
    auto by_type = [&](auto dim) {
        const bool u32 = U && u_precision == IBAMR_FP32C;
        if (f_precision == IBAMR_FP64)
            u32 ? go(dim, 0.0, 0.0f) : go(dim, 0.0, 0.0);
        else
            u32 ? go(dim, 0.0f, 0.0f) : go(dim, 0.0f, 0.0);
    };
    if (f->ndim == 3)
        by_type(std::integral_constant<int, 3>());
    else
        by_type(std::integral_constant<int, 2>());
    F_HIP(hipGetLastError());
    return IBAMR_OK;
}

} // extern "C"
