// Objective, sensitivities, density filters and the optimality-criteria update on the device.
//
//   unit compliance     TopOpti_ComputeUnitCompliance(_Super)   TOP_GPU.m:580-600, 2622-2645
//   sub-voxel energies  pre_compute_der                         TOP_GPU.m:2646-2671
//   SIMP / dc           TOP_GPU.m:168-174, 189-209
//   OC update           TOP_GPU.m:233-253 (bisection on the device, deterministic reductions)
//   PDE filter          TopOpti_SetupPDEfilter_matrixFree / ConductPDEFiltering / MatTimesVec_matrixFree_B
//                       TOP_GPU.m:880-1031 (nodal Helmholtz solve with Jacobi-PCG)
//   convolution filter  imfilter density filter of super-element mode, TOP_GPU.m:112-121, 220-227, 262-265
#include <cmath>
#include <cstring>
#include <memory>
#include <mutex>

#include "kernels.h"
#include "model.h"
#include "pcg.h"
#include "scratch.h"
#include "solver.h"
#include "topopt.h"

namespace tg {
namespace {

// ce_e = u_e' * Ke * u_e; u is a full-grid interleaved vector; output in solid-element order.
__global__ void k_unit_compliance(const double *__restrict__ u, const double *__restrict__ K0,
                                  const int32_t *__restrict__ eleFull0, int64_t Ne, const Grid g, double *__restrict__ ce) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= Ne) return;
    const int64_t e = eleFull0[k];
    const int ey = (int)(e % g.EY), ex = (int)((e / g.EY) % g.EX), ez = (int)(e / ((int64_t)g.EY * g.EX));
    double ue[24];
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const int64_t m = (ey + vtx_y(b)) + (int64_t)g.NY * ((ex + vtx_x(b)) + (int64_t)g.NX * (ez + vtx_z(b)));
        ue[3 * b] = u[3 * m];
        ue[3 * b + 1] = u[3 * m + 1];
        ue[3 * b + 2] = u[3 * m + 2];
    }
    double s = 0;
    for (int j = 0; j < 24; ++j) {
        double kj = 0;
#pragma unroll
        for (int i = 0; i < 24; ++i) kj += ue[i] * K0[i + 24 * j];  // (u_e' * Ke)_j
        s += kj * ue[j];
    }
    ce[k] = s;
}

// Super-element mode: ce_e = u_e' K_mat_e u_e, K_mat entry-major.  Eight threads per element, three columns each,
// their sums added in column order: consecutive threads read consecutive elements' entries, and a chain of
// 72 loads replaces one of 576 (160 us at 6,000 elements with a thread per element, 46 this way).
constexpr int UC_PARTS = 8, UC_ELEMS = 32;
__global__ __launch_bounds__(UC_PARTS * UC_ELEMS) void k_unit_compliance_super(const double *__restrict__ u,
                                                                               const double *__restrict__ Km, int64_t ldk,
                                                                               const int32_t *__restrict__ eleFull0,
                                                                               int64_t Ne, const Grid g,
                                                                               double *__restrict__ ce) {
    __shared__ double part[UC_PARTS][UC_ELEMS];
    const int el = threadIdx.x % UC_ELEMS, p = threadIdx.x / UC_ELEMS;
    const int64_t k = (int64_t)blockIdx.x * UC_ELEMS + el;
    const int64_t e = eleFull0[k < Ne ? k : Ne - 1];
    const int ey = (int)(e % g.EY), ex = (int)((e / g.EY) % g.EX), ez = (int)(e / ((int64_t)g.EY * g.EX));
    double ue[24];
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const int64_t m = (ey + vtx_y(b)) + (int64_t)g.NY * ((ex + vtx_x(b)) + (int64_t)g.NX * (ez + vtx_z(b)));
        ue[3 * b] = u[3 * m];
        ue[3 * b + 1] = u[3 * m + 1];
        ue[3 * b + 2] = u[3 * m + 2];
    }
    double s = 0;
#pragma unroll
    for (int b = 0; b < UC_PARTS; ++b)  // (static indices into ue)
        if (p == b)
#pragma unroll
            for (int j = 3 * b; j < 3 * b + 3; ++j) {
                double kj = 0;
#pragma unroll
                for (int i = 0; i < 24; ++i) kj += Km[(int64_t)(j + 24 * i) * ldk + e] * ue[i];  // (K_mat_e u_e)_j
                s += kj * ue[j];
            }
    part[p][el] = s;
    __syncthreads();
    if (p == 0 && k < Ne) {
        for (int b = 1; b < UC_PARTS; ++b) s += part[b][el];
        ce[k] = s;
    }
}

// dc(q, e) = u_e' I_q u_e = sum over i <= j of (I_q(i, j) + I_q(j, i)) u_i u_j (half of it for i = j): a product of
// the 64 x 300 sub-voxel coefficients with the element's 300 products u_i u_j, on the matrix cores (f64 16x16x4:
// 16 sub-voxels x 4 products x 16 elements; layouts as in the solver's Galerkin product).  A wavefront has 16
// elements, their displacements in LDS, and forms its products as it goes; the four wavefronts of a workgroup
// take a quarter of the products each and add up in wavefront order.  Sub-voxel tiles are stored element by
// element.  330 us at 6,000 elements with a thread per element and sub-voxel, 47 here.
typedef double tg_tdbl4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void k_subvoxel_energy(const double *__restrict__ u, const double *__restrict__ Imat,
                                                         const int32_t *__restrict__ eleFull0, int64_t Ne, const Grid g,
                                                         double *__restrict__ dc) {
    __shared__ double su[24][17];
    __shared__ double red[4][16][65];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
    const int64_t k0 = (int64_t)blockIdx.x * 16;
    for (int i = threadIdx.x; i < 128; i += 256) {  // one vertex of one element
        const int el = i & 15, b = i >> 4;
        const int64_t e = eleFull0[k0 + el < Ne ? k0 + el : Ne - 1];
        const int ey = (int)(e % g.EY), ex = (int)((e / g.EY) % g.EX), ez = (int)(e / ((int64_t)g.EY * g.EX));
        const int64_t m = (ey + vtx_y(b)) + (int64_t)g.NY * ((ex + vtx_x(b)) + (int64_t)g.NX * (ez + vtx_z(b)));
        for (int c = 0; c < 3; ++c) su[3 * b + c][el] = u[3 * m + c];
    }
    __syncthreads();
    tg_tdbl4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = tg_tdbl4{0.0, 0.0, 0.0, 0.0};
    // products 4 kk + lk of the packed upper triangle, p = i + j (j + 1) / 2; 75 groups of four
    const int kk0 = w * 19, kk1 = min(kk0 + 19, 75);
    int p = 4 * kk0 + lk, j = (int)((sqrtf(8.0f * (float)p + 1.0f) - 1.0f) * 0.5f);
    if (ksym_index(0, j) > p) --j;
    if (ksym_index(0, j + 1) <= p) ++j;
    int i = p - ksym_index(0, j);
    for (int kk = kk0; kk < kk1; ++kk) {
        const double b = su[i][li] * su[j][li];
        double a[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const double *I = Imat + (size_t)576 * (16 * t + li);
            a[t] = i == j ? I[25 * i] : I[i + 24 * j] + I[j + 24 * i];
        }
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t], b, acc[t], 0, 0, 0);
        for (i += 4; i > j; ++j) i -= j + 1;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) red[w][li][16 * t + 4 * r + lk] = acc[t][r];
    __syncthreads();
    for (int idx = threadIdx.x; idx < 1024; idx += 256) {
        const int el = idx >> 6, q = idx & 63;
        if (k0 + el >= Ne) continue;
        double s = red[0][el][q];
        for (int v = 1; v < 4; ++v) s += red[v][el][q];
        dc[64 * (k0 + el) + q] = s;
    }
}

__global__ void k_simp(const double *__restrict__ x, double *__restrict__ E, int64_t n, double Emin, double E0,
                       double p) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) E[i] = Emin + pow(x[i], p) * (E0 - Emin);
}

// dc = -(p (E0 - Emin) x^(p-1)) .* (ce / cSolid)
__global__ void k_sens(const double *__restrict__ x, const double *__restrict__ ce, double *__restrict__ dc,
                       int64_t n, int per, double Emin, double E0, double p, double cSolid) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dc[i] = -(p * (E0 - Emin) * pow(x[i], p - 1)) * (ce[i / per] / cSolid);
}

__global__ void k_mul(const double *__restrict__ a, const double *__restrict__ b, double *__restrict__ c, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) c[i] = a[i] * b[i];
}

__global__ void k_div_floor(const double *__restrict__ a, const double *__restrict__ x, double *__restrict__ c,
                            double fl, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) c[i] = a[i] / fmax(fl, x[i]);
}

// c = (b != 0) ? v : a  (xPhys(passiveElements) = 1 after the density filter, TOP_GPU.m:270, 273)
__global__ void k_set_where(const double *__restrict__ a, const double *__restrict__ b, double *__restrict__ c, double v,
                            int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) c[i] = b[i] != 0.0 ? v : a[i];
}

// c = a + v b  (the load cases' weighted sum of unit compliances, ceList * objWeightingList_,
// TOP_GPU.m:599, 2644, 2671); c may be a (no restrict: each entry is read before it is written)
__global__ void k_axpy(const double *a, const double *__restrict__ b, double *c, double v, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) c[i] = a[i] + v * b[i];
}

// ---- reductions ------------------------------------------------------------------------------
enum { R_SUM = 0, R_DOT = 1, R_MAXABSDIFF = 2, R_SHARP = 3 };

template <int OP>
__global__ __launch_bounds__(RED_THREADS) void k_red_partial(const double *__restrict__ a, const double *__restrict__ b,
                                                             int64_t n, double *__restrict__ partial) {
    const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;
    const int64_t lo = (int64_t)blockIdx.x * chunk, hi = lo + chunk < n ? lo + chunk : n;
    double s = 0;
    for (int64_t i = lo + threadIdx.x; i < hi; i += blockDim.x) {
        if (OP == R_SUM) s += a[i];
        else if (OP == R_DOT) s += a[i] * b[i];
        else if (OP == R_SHARP) s += a[i] * (1.0 - a[i]);
        else s = fmax(s, fabs(a[i] - b[i]));
    }
    __shared__ double sh[RED_THREADS];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = RED_THREADS / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] = OP == R_MAXABSDIFF ? fmax(sh[threadIdx.x], sh[threadIdx.x + w])
                                                                      : sh[threadIdx.x] + sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

// host, seq: the result in pinned host memory, and the number published after it (Scratch::wait)
template <int OP>
__global__ __launch_bounds__(RED_THREADS) void k_red_final(const double *__restrict__ partial, int nb,
                                                           double *__restrict__ host, unsigned long long *seq_ptr,
                                                           unsigned long long seq) {
    __shared__ double sh[RED_THREADS];
    double s = 0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) s = OP == R_MAXABSDIFF ? fmax(s, partial[i]) : s + partial[i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int w = RED_THREADS / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] = OP == R_MAXABSDIFF ? fmax(sh[threadIdx.x], sh[threadIdx.x + w])
                                                                      : sh[threadIdx.x] + sh[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        *host = sh[0];
        __hip_atomic_store(seq_ptr, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ---- optimality criteria ---------------------------------------------------------------------
__device__ inline bool oc_open(double l1, double l2) { return (l2 - l1) / (l1 + l2) > 1e-6; }

__device__ inline double oc_xnew(double x, double dc, double dv, double lmid, double move) {
    return fmax(0.0, fmax(x - move, fmin(1.0, fmin(x + move, x * sqrt(-dc / dv / lmid)))));
}

// The bisection on the multiplier, OC_DEPTH steps a launch.  From a bracket (l1, l2) those steps can meet
// 2^OC_DEPTH - 1 midpoints, a binary tree (node 1 the middle; from node m to 2 m + 1 where gt > 0, l1 = mid, else to
// 2 m): every launch sums xnew - x for all of them over one pass of the data, and the next launch's workgroups each
// walk the tree with the finished sums, to the bracket that the same steps one by one would reach.  A pass needs x and
// b = x sqrt(-dc / dv), so a midpoint costs a product with 1 / sqrt(mid) and the clamps; k_oc_apply evaluates the update
// itself at the last midpoint.
// b is kept in xnew until that is written, but only where the bisection is known to end: a call that fails leaves
// the caller's array as it was.  The bracket closes within 19 steps of the first gt > 0, and gt does not increase with
// the multiplier (nor do its rounded sums, in one fixed order), so gt > 0 at OC_FLOOR, the midpoint that is reached after 397
// steps of l1 = 0, says that it closes within the 416 steps there are.  The first pass sums for OC_FLOOR too, the
// second one decides and writes b (at 4.2 million entries 35 and 40 us, the later ones 30); where it may not (or the
// caller's arrays overlap), every pass forms b itself.
// passive (may be null): entries with a nonzero indicator take xnew = 1 inside every step, so
// they enter gt (xnew(passiveElements) = 1.0, TOP_GPU.m:239, 247).
// Bound by the passes' two streams on large designs and by launches on small ones: 16 passes for 64 steps, 30 us each
// at 4.2 million entries and 11 at 27,648, against 64 steps of two launches each, 21.6 us (17 and 4.6) and 6.2 a step.
constexpr int OC_DEPTH = 4, OC_NODES = (1 << OC_DEPTH) - 1, OC_BLOCKS = 512;
constexpr double OC_FLOOR = 1e9 * 0x1p-397;
struct OcState {
    double l1, l2, lmid, steps;  // bracket, the last executed step's midpoint, steps executed
    double keep;                 // whether xnew holds b
};

// The state after the steps that the sums decide; sums[m - 1]: node m's sum of xnew - x.
__device__ inline OcState oc_walk(OcState s, const double *sums, double fval, double n) {
    int node = 1;
    for (int k = 0; k < OC_DEPTH && oc_open(s.l1, s.l2); ++k) {
        s.lmid = 0.5 * (s.l2 + s.l1);
        const bool up = fval + sums[node - 1] / n > 0;
        if (up) s.l1 = s.lmid;
        else s.l2 = s.lmid;
        s.steps += 1;
        node = 2 * node + (up ? 1 : 0);
    }
    return s;
}

// old: the state that the previous launch's sums (partial_in, nb rows) refine; now: where the result goes.
// PASS: 0 the first, 1 the second, 2 any later one.  b (may be null): where b may be kept.
template <int PASS>
__global__ __launch_bounds__(RED_THREADS) void k_oc_pass(const double *__restrict__ x, const double *__restrict__ dc,
                                                         const double *__restrict__ dv, double *__restrict__ b,
                                                         const double *__restrict__ passive, int64_t n, double fval,
                                                         double move, const OcState *__restrict__ old,
                                                         OcState *__restrict__ now, const double *__restrict__ partial_in,
                                                         double *__restrict__ partial_out) {
    constexpr int NIN = OC_NODES + (PASS == 1), NOUT = OC_NODES + (PASS == 0);  // the last of them: OC_FLOOR's
    __shared__ double sh[4][OC_NODES + 1], sums[OC_NODES + 1], scale[OC_NODES + 1];
    __shared__ OcState st;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, nb = gridDim.x;
    auto reduce = [&](double *v, int count) {  // over the workgroup, in a fixed order; in sums
#pragma unroll
        for (int k = 0; k < OC_NODES + 1; ++k)
            if (k < count) {
                for (int o = 32; o > 0; o >>= 1) v[k] += __shfl_down(v[k], o, 64);
                if (lane == 0) sh[w][k] = v[k];
            }
        __syncthreads();
        if (t < count) sums[t] = (sh[0][t] + sh[1][t]) + (sh[2][t] + sh[3][t]);
        __syncthreads();
    };
    double acc[OC_NODES + 1];
#pragma unroll
    for (int k = 0; k < OC_NODES + 1; ++k) acc[k] = 0.0;
    if (PASS > 0) {
        for (int r = t; r < nb; r += RED_THREADS)
#pragma unroll
            for (int k = 0; k < NIN; ++k) acc[k] += partial_in[(int64_t)k * nb + r];
        reduce(acc, NIN);
    }
    if (t == 0) {
        st = PASS == 0 ? OcState{0.0, 1e9, 0.0, 0.0, 0.0} : oc_walk(*old, sums, fval, (double)n);
        if (PASS == 1) st.keep = b && fval + sums[OC_NODES] / (double)n > 0 ? 1.0 : 0.0;
        if (blockIdx.x == 0) *now = st;
    }
    __syncthreads();
    if (!oc_open(st.l1, st.l2)) return;
    if (t < OC_NODES) {  // node t + 1: its path from the root gives its bracket
        double l1 = st.l1, l2 = st.l2;
        const int node = t + 1, depth = 31 - __clz(node);
        for (int k = depth - 1; k >= 0; --k) {
            const double mid = 0.5 * (l2 + l1);
            if ((node >> k) & 1) l1 = mid;
            else l2 = mid;
        }
        scale[t] = 1.0 / sqrt(0.5 * (l2 + l1));
    } else if (t == OC_NODES) {
        scale[t] = 1.0 / sqrt(OC_FLOOR);
    }
    __syncthreads();
    double sc[NOUT];
#pragma unroll
    for (int k = 0; k < NOUT; ++k) {
        sc[k] = scale[k];
        acc[k] = 0.0;
    }
    const int64_t stride = (int64_t)nb * RED_THREADS;
    auto sweep = [&](auto root) {  // root(i, x): b of entry i
#pragma unroll 2
        for (int64_t i = (int64_t)blockIdx.x * RED_THREADS + t; i < n; i += stride) {
            const double xi = x[i], bi = root(i, xi);
            double lo = fmax(0.0, xi - move), hi = fmin(1.0, xi + move);
            if (passive && passive[i] != 0.0) lo = hi = 1.0;
#pragma unroll
            for (int k = 0; k < NOUT; ++k) acc[k] += fmax(lo, fmin(hi, bi * sc[k])) - xi;
        }
    };
    auto form = [&](int64_t i, double xi) { return xi * sqrt(-dc[i] / dv[i]); };
    if (PASS == 0 || st.keep == 0.0) sweep(form);
    else if (PASS == 1) sweep([&](int64_t i, double xi) { return b[i] = form(i, xi); });
    else sweep([&](int64_t i, double) { return b[i]; });
    reduce(acc, NOUT);
    if (t < NOUT) partial_out[(int64_t)t * nb + blockIdx.x] = sums[t];
}

// The state after the last pass, for the host's check (and the apply's midpoint).
__global__ __launch_bounds__(RED_THREADS) void k_oc_close(int64_t n, double fval, const OcState *__restrict__ old,
                                                          OcState *__restrict__ now, const double *__restrict__ partial,
                                                          int nb, double *__restrict__ host, unsigned long long *seq_ptr,
                                                          unsigned long long seq) {
    __shared__ double sums[OC_NODES];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int k = w; k < OC_NODES; k += RED_THREADS / 64) {
        double s = 0;
        for (int r = lane; r < nb; r += 64) s += partial[(int64_t)k * nb + r];
        for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
        if (lane == 0) sums[k] = s;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const OcState s = oc_walk(*old, sums, fval, (double)n);
        *now = s;
        *(OcState *)host = s;
        __hip_atomic_store(seq_ptr, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// xnew, and each workgroup's max |xnew - x|
__global__ __launch_bounds__(RED_THREADS) void k_oc_apply(const double *__restrict__ x, const double *__restrict__ dc,
                                                          const double *__restrict__ dv, const double *__restrict__ passive,
                                                          double *xnew, int64_t n, double move,
                                                          const OcState *__restrict__ st, double *__restrict__ partial) {
    __shared__ double sh[RED_THREADS];
    const double lmid = st->lmid;
    double m = 0;
    for (int64_t i = (int64_t)blockIdx.x * RED_THREADS + threadIdx.x; i < n; i += (int64_t)gridDim.x * RED_THREADS) {
        const double xi = x[i];
        const double v = passive && passive[i] != 0.0 ? 1.0 : oc_xnew(xi, dc[i], dv[i], lmid, move);
        xnew[i] = v;
        m = fmax(m, fabs(v - xi));
    }
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int w = RED_THREADS / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) sh[threadIdx.x] = fmax(sh[threadIdx.x], sh[threadIdx.x + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

// ---- PDE filter ------------------------------------------------------------------------------
// The filter's Jacobi-PCG has two kernels an iteration.  k_filter_step makes the direction p = inv r +
// beta p, adds the previous step to the iterate and applies the operator to the new direction;
// k_filter_update takes the residual on.  Each finishes the other's partial sums in all its workgroups (one
// order, one value), and workgroup 0 of the next k_filter_step tells the host the residual norm, so the
// host's look at it runs beside that kernel: when the loop stops there, that launch has only made the last
// update of the iterate, which is due anyway.
constexpr int FS_THREADS = 512;

// The solid elements around each node, one bit each: (oy+1) + 2(ox+1) + 4(oz+1) for offsets in {-1, 0}.
__global__ void k_filter_codes(const uint8_t *__restrict__ eleMask, const Grid g, uint8_t *__restrict__ code) {
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= g.nodes()) return;
    const int iy = (int)(n % g.NY);
    const int64_t t = n / g.NY;
    const int ix = (int)(t % g.NX), iz = (int)(t / g.NX);
    int c = 0;
    for (int j = 0; j < 8; ++j) {
        const int ey = iy - 1 + (j & 1), ex = ix - 1 + ((j >> 1) & 1), ez = iz - 1 + (j >> 2);
        if ((unsigned)ey < (unsigned)g.EY && (unsigned)ex < (unsigned)g.EX && (unsigned)ez < (unsigned)g.EZ &&
            eleMask[ey + (int64_t)g.EY * (ex + (int64_t)g.EX * ez)])
            c |= 1 << j;
    }
    code[n] = (uint8_t)c;
}

// The sums of a and of b over the workgroup (whole wavefronts, at most 16), in every thread.
__device__ inline void block_sum2(double &a, double &b) {
    __shared__ double sh[32];
    for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
    }
    __syncthreads();  // the last use of the shared array is over
    if ((threadIdx.x & 63) == 0) {
        sh[threadIdx.x >> 6] = a;
        sh[16 + (threadIdx.x >> 6)] = b;
    }
    __syncthreads();
    a = b = 0;
    for (int w = 0; w < (int)blockDim.x >> 6; ++w) {
        a += sh[w];
        b += sh[16 + w];
    }
}

// element -> node: r_n = b_n = sum over solid elements around n of src_e * (1/8)  (TOP_GPU.m:975-996), with
// partial sums of b.b and of the preconditioned b.(inv b).  A chain of three loads a node (its elements, their
// numbers, their values): the workgroups are the widest there are, so that few nodes of a thread follow each
// other (128x256x128: 45 us; of 256
// threads, with a branch an element, 98)
constexpr int E2N_THREADS = 1024;
__global__ __launch_bounds__(E2N_THREADS) void k_e2n(const double *__restrict__ src, const int32_t *__restrict__ eleFwd,
                                                     const uint8_t *__restrict__ code, const Grid g,
                                                     const double *__restrict__ inv, double *__restrict__ r,
                                                     double *__restrict__ pbb, double *__restrict__ pzr) {
    double bb = 0, zr = 0;
    const unsigned nn = (unsigned)g.nodes(), NY = g.NY, NX = g.NX;  // node numbers are 32 bits (the maps')
    for (unsigned n = blockIdx.x * E2N_THREADS + threadIdx.x; n < nn; n += gridDim.x * E2N_THREADS) {
        double s = 0;
        const int c = code[n];
        if (c) {
            const unsigned t = n / NY, iy = n - t * NY, iz = t / NX, ix = t - iz * NX;
            const int e0 = (int)(iy - 1 + g.EY * (ix - 1 + g.EX * (iz - 1)));
            auto at = [&](int j) { return e0 + (j & 1) + g.EY * (((j >> 1) & 1) + g.EX * (j >> 2)); };
            const int ok = at(__ffs(c) - 1);  // an element that is there, in place of those that are not: no branches
            int32_t k[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) k[j] = eleFwd[c & (1 << j) ? at(j) : ok];
            double v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = src[k[j] - 1];
#pragma unroll
            for (int j = 0; j < 8; ++j) s += c & (1 << j) ? v[j] * (1.0 / 8) : 0.0;
        }
        r[n] = s;
        bb += s * s;
        zr += inv[c] * s * s;
    }
    block_sum2(bb, zr);
    if (threadIdx.x == 0) {
        pbb[blockIdx.x] = bb;
        pzr[blockIdx.x] = zr;
    }
}

struct FilterStep {
    Grid g;
    int ty, tx, tyn, chunk;        // nodes of a tile along y and x, tiles along y, planes of a chunk
    double k0, k1, k2, k3;         // the element matrix: entries between corners 0, 1, 2 and 3 edges apart
    const uint8_t *code;
    const double *inv, *r;
    double *pold, *p, *y, *v;      // the last direction, the new one, the iterate, the product
    const double *prr, *pzr;       // the partial sums r.r (b.b at first) and z.r that k_filter_update left
    int np;
    double *ppv;                   // the partial sums p.v for it
    double *scal, *host;
    unsigned long long seq;        // published with the residual norm
    int xo, xn;                    // slots of z.r: the last direction's and this one's
};

// p = inv r + beta p;  y += lambda p of before;  v_n = sum over solid elements around n of (K p_e)_a
// (MatTimesVec_matrixFree_B, TOP_GPU.m:1008-1031);  partial sums of p.v.   IT: 0 the first direction, 1 the
// second (the iterate is still zero), 2 any later one.
// A workgroup walks a tile of columns up z, a thread a column (the tile's rim only supplies its p to the
// neighbours through LDS), with the next plane's loads in flight.  The element matrix has one entry per
// distance of two corners, so a plane's part of an element's product is a sum over the quadrant of the 3x3
// nodes around the column, and a layer of elements is two such parts: each plane is read and turned once.
// Bound by memory: six streams of 8 bytes per node and the rims (128x256x128: 63 us, 3.3 TB/s without the
// rims; with k_filter_update's 19 an iteration takes 82 us, where nine launches took 200; 24x48x24: 6.6 and
// 4.7 us).  512 threads a tile: 256 take 72 us, more of them being rim, and 1024 take 61 but 9.5 at 24x48x24.
template <int IT>
__global__ __launch_bounds__(FS_THREADS) void k_filter_step(const FilterStep a) {
    __shared__ double pl[2][FS_THREADS], tab[256];
    const Grid &g = a.g;
    const int t = threadIdx.x, h = a.ty + 2;
    if (t < 256) tab[t] = a.inv[t];
    double rr = 0, zr = 0;
    for (int i = t; i < a.np; i += FS_THREADS) {
        rr += a.prr[i];
        zr += a.pzr[i];
    }
    block_sum2(rr, zr);  // its barriers cover tab too
    double beta = 0, lam = 0;
    if (IT) {
        const double zr0 = a.scal[a.xo];
        beta = zr / zr0;
        lam = zr0 / a.scal[S_PV];
    }
    if (blockIdx.x == 0 && blockIdx.y == 0 && t == 0) {
        a.scal[a.xn] = zr;  // the other slot: every workgroup reads the old one
        if (IT == 0) {
            a.scal[S_BB] = rr;
        } else {
            a.host[S_BB] = a.scal[S_BB];
            a.host[S_RR] = rr;
            __hip_atomic_store((unsigned long long *)(a.host + 16), a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    const int ly = t % h, lx = t / h;
    const int iy = (int)(blockIdx.x % a.tyn) * a.ty + ly - 1, ix = (int)(blockIdx.x / a.tyn) * a.tx + lx - 1;
    const bool on = lx < a.tx + 2 && (unsigned)iy < (unsigned)g.NY && (unsigned)ix < (unsigned)g.NX;
    const bool own = on && ly >= 1 && ly <= a.ty && lx >= 1 && lx <= a.tx;
    const int64_t plane = (int64_t)g.NY * g.NX;
    const int z0 = (int)blockIdx.y * a.chunk, z1 = min(z0 + a.chunk, g.NZ);
    const int zb = max(z0 - 1, 0), ze = min(z1, g.NZ - 1);  // planes read
    int64_t n = iy + (int64_t)g.NY * ix + plane * zb;
    double r = 0, po = 0, y = 0;
    int c = 0;
    auto load = [&](int z, int64_t m) {
        if (!on) return;
        c = a.code[m];
        r = a.r[m];
        if (IT) po = a.pold[m];
        if (IT == 2 && own && z >= z0 && z < z1) y = a.y[m];
    };
    load(zb, n);
    double q1[4] = {}, q2[4] = {}, acc = 0, pc = 0, pv = 0;  // of the plane below
    int cc = 0;
    for (int z = zb; z <= ze; ++z, n += plane) {
        const double p = IT ? tab[c] * r + beta * po : tab[c] * r, p0 = po, y0 = y;
        const int cz = c;
        if (z < ze) load(z + 1, n + plane);
        double *b = pl[z & 1];
        b[t] = p;
        const bool in = own && z >= z0 && z < z1;
        if (in) {
            a.p[n] = p;
            if (IT) a.y[n] = (IT == 2 ? y0 : 0.0) + lam * p0;
        }
        __syncthreads();
        if (!own) continue;
        const double up = b[t + 1], dn = b[t - 1], lf = b[t - h], rt = b[t + h];
        const double f[4] = {dn + lf, up + lf, dn + rt, up + rt};
        const double d[4] = {b[t - 1 - h], b[t + 1 - h], b[t - 1 + h], b[t + 1 + h]};
        double below = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const double e1 = a.k0 * p + a.k1 * f[k] + a.k2 * d[k], e2 = a.k1 * p + a.k2 * f[k] + a.k3 * d[k];
            if (cc & (16 << k)) {  // the element between the two planes: above the last, below this one
                acc += q1[k] + e2;
                below += e1 + q2[k];
            }
            q1[k] = e1;
            q2[k] = e2;
        }
        if (z > z0) {  // the plane below is complete (z0 - 1 is another chunk's)
            a.v[n - plane] = acc;
            pv += pc * acc;
        }
        acc = below;
        pc = p;
        cc = cz;
    }
    if (own && z1 == g.NZ) {  // the top plane has no layer above
        a.v[n - plane] = acc;
        pv += pc * acc;
    }
    double unused = 0;
    block_sum2(pv, unused);
    if (t == 0) a.ppv[blockIdx.x + gridDim.x * blockIdx.y] = pv;
}

// r -= lambda v, with partial sums of r.r and r.(inv r); p.v is finished here from k_filter_step's partials.
__global__ __launch_bounds__(RED_THREADS) void k_filter_update(double *__restrict__ r, const double *__restrict__ v,
                                                               int64_t n, const uint8_t *__restrict__ code,
                                                               const double *__restrict__ inv,
                                                               const double *__restrict__ ppv, int npv,
                                                               double *__restrict__ scal, int ix,
                                                               double *__restrict__ prr, double *__restrict__ pzr) {
    __shared__ double tab[256];
    tab[threadIdx.x] = inv[threadIdx.x];
    double pv = 0, zr = 0, rr = 0;
    for (int i = threadIdx.x; i < npv; i += RED_THREADS) pv += ppv[i];
    block_sum2(pv, zr);
    if (blockIdx.x == 0 && threadIdx.x == 0) scal[S_PV] = pv;
    const double lam = scal[ix] / pv;
    zr = 0;
    for (int64_t i = (int64_t)blockIdx.x * RED_THREADS + threadIdx.x; i < n; i += (int64_t)gridDim.x * RED_THREADS) {
        const double x = r[i] - lam * v[i];
        r[i] = x;
        rr += x * x;
        zr += tab[code[i]] * x * x;
    }
    block_sum2(rr, zr);
    if (threadIdx.x == 0) {
        prr[blockIdx.x] = rr;
        pzr[blockIdx.x] = zr;
    }
}

// node -> element: tar_e = sum(tar(eNod(e,:))) * (1/8)  (TOP_GPU.m:1004-1005)
__global__ void k_n2e(const double *__restrict__ tar, const int32_t *__restrict__ eleFull0, int64_t Ne, const Grid g,
                      double *__restrict__ out) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= Ne) return;
    const unsigned e = eleFull0[k], EY = g.EY, EX = g.EX;
    const unsigned c = e / EY, ey = e - c * EY, ez = c / EX, ex = c - ez * EX;
    double s = 0;
#pragma unroll
    for (int b = 0; b < 8; ++b)
        s += tar[(ey + vtx_y(b)) + (int64_t)g.NY * ((ex + vtx_x(b)) + (int64_t)g.NX * (ez + vtx_z(b)))];
    out[k] = s * (1.0 / 8);
}

// ---- convolution filter ----------------------------------------------------------------------
// grid voxel (iy, ix, iz) of the num-times refined box <-> element-major index q + num^3 * element
__device__ inline int64_t cv_new_index(int iy, int ix, int iz, int num, int Y, int X) {
    const int64_t big = iy / num + (int64_t)Y * (ix / num + (int64_t)X * (iz / num));
    const int64_t loc = iy % num + num * (ix % num + num * (iz % num));
    return loc + (int64_t)num * num * num * big;
}

// out[p] = sum_q h(q) * in(p + q - c) on a zero-padded grid (imfilter, 'same', bcF = 0), in = src, for the adjoint
// src ./ Hs, or ones for Hs itself, read where the caller has it: a call leaves nothing in the handle, so calls on one
// handle may overlap (threads, replays of a captured call).
// MODE 0: out = result ./ Hs  (forward: xPhys = imfilter(x)./Hs)   MODE 1: out = result  (adjoint: imfilter(dc./Hs))
// MODE 2: out = result on the grid  (Hs = imfilter(1))
template <int MODE>
__device__ __forceinline__ void conv_store(double *__restrict__ out, const double *__restrict__ Hs, int iy, int ix, int iz,
                                           int GY, int GX, int num, int Y, int X, double s) {
    const int64_t p = iy + (int64_t)GY * (ix + (int64_t)GX * iz);
    if (MODE == 0) out[cv_new_index(iy, ix, iz, num, Y, X)] = s / Hs[p];
    else if (MODE == 1) out[cv_new_index(iy, ix, iz, num, Y, X)] = s;
    else out[p] = s;
}

// cv_new_index is a sum of one term per axis; this is that term of one axis, voxel by voxel (loc: between voxels of an
// element, big: between elements).
struct CvAxis {
    int64_t off, loc, skip;
    int rem, num;
    __device__ CvAxis(int i, int n, int64_t l, int64_t big)
        : off(i / n * big + i % n * l), loc(l), skip(big - (n - 1) * l), rem(i % n), num(n) {}
    __device__ void next() {
        const bool last = ++rem == num;
        off += last ? skip : loc;
        rem = last ? 0 : rem;
    }
};

// Cones of 1 to CONV_HR voxels' reach.  The cone is even in each direction: the planes z - dz and z + dz are added
// as they are staged, which halves the products.  A workgroup has LY x LX blocks of CONV_Y voxels along y in
// one plane, a block to a lane, and its four wavefronts share out the dz (0, 7, 8, ..; 1, 6, 9, ..; so that the
// wide and the narrow discs of the ball fall together), each with a plane of its own in LDS and no barrier but
// for the sum at the end.  Per row (dx, dz) of the cone a lane reads CONV_Y + 2 HR values of a column into registers
// for up to CONV_Y (2 HR + 1) products, over the taps with a weight only (lim: the last such dy, uniform).
// Bound by LDS reads and FP64 products together: 56 us (forward) and 67 (adjoint, which divides every value as it stages
// it) for the 40 x 240 x 40 sub-voxels of a 10 x 60 x 10 beam at a reach of 6, against 670 and 930 with a thread per
// voxel that walked the whole cube and found each tap's address by division.
constexpr int CONV_Y = 8, CONV_HR = 12;
template <int HR, int MODE>
__global__ __launch_bounds__(256) void k_conv(const double *__restrict__ src, const double *__restrict__ Hs,
                                              const double *__restrict__ h, const int32_t *__restrict__ lim, int GY, int GX,
                                              int GZ, int num, int Y, int X, int LY, int LX, int pitch,
                                              double *__restrict__ out) {
    extern __shared__ double sm[];
    constexpr int W = HR + 1;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int tilesY = (GY + CONV_Y * LY - 1) / (CONV_Y * LY);
    const int y0 = (int)(blockIdx.x % tilesY) * CONV_Y * LY, x0 = (int)(blockIdx.x / tilesY) * LX, iz = blockIdx.y;
    const int rows = CONV_Y * LY + 2 * HR, cols = LX + 2 * HR;
    double *plane = sm + w * cols * pitch;
    const int ly = lane % LY, lx = lane / LY;
    const double *mine = plane + (lx < LX ? lx : 0) * pitch + CONV_Y * ly;
    double acc[CONV_Y] = {};
    for (int k = 0;; ++k) {
        const int dz = 4 * k + ((k & 1) ? 3 - w : w);
        if (4 * k > HR) break;
        if (dz > HR) continue;
        const int zl = iz - dz, zh = iz + dz;
        const bool okl = zl >= 0, okh = dz > 0 && zh < GZ;
        const int64_t n3 = (int64_t)num * num * num, layer = n3 * Y * X;
        const double *sl = src + (okl ? CvAxis(zl, num, num * num, layer).off : 0);
        const double *sh = src + (okh ? CvAxis(zh, num, num * num, layer).off : 0);
        const double *Hl = Hs + (int64_t)GY * GX * (okl ? zl : 0), *Hh = Hs + (int64_t)GY * GX * (okh ? zh : 0);
        for (int yy = lane; yy < rows; yy += 64) {
            const int y = y0 - HR + yy;
            const bool oky = (unsigned)y < (unsigned)GY;
            const CvAxis ay(oky ? y : 0, num, 1, n3);
            CvAxis ax(max(x0 - HR, 0), num, num, n3 * Y);
            for (int xx = 0; xx < cols; ++xx) {
                const int x = x0 - HR + xx;
                double v = 0.0;
                if ((unsigned)x < (unsigned)GX) {
                    if (oky) {
                        const int64_t at = ax.off + ay.off, p = y + (int64_t)GY * x;
                        if (okl) v = MODE == 2 ? 1.0 : MODE == 1 ? sl[at] / Hl[p] : sl[at];
                        if (okh) v += MODE == 2 ? 1.0 : MODE == 1 ? sh[at] / Hh[p] : sh[at];
                    }
                    ax.next();
                }
                plane[xx * pitch + yy] = v;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int dx = -HR; dx <= HR; ++dx) {
            const int row = dz * W + (dx < 0 ? -dx : dx), last = lim[row];
            if (last < 0) continue;
            const double *c = mine + (HR + dx) * pitch;
            double v[CONV_Y + 2 * HR];
#pragma unroll
            for (int i = 0; i < CONV_Y + 2 * HR; ++i) v[i] = c[i];
#pragma unroll
            for (int i = 0; i <= HR; ++i) {
                if (i <= last) {
                    const double hv = h[row * W + i];
#pragma unroll
                    for (int o = 0; o < CONV_Y; ++o) {
                        acc[o] += hv * v[o + HR - i];
                        if (i > 0) acc[o] += hv * v[o + HR + i];
                    }
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();  // the planes are done with
#pragma unroll
    for (int o = 0; o < CONV_Y; ++o) sm[(w * CONV_Y + o) * 64 + lane] = acc[o];
    __syncthreads();
    if (lx >= LX) return;
#pragma unroll
    for (int k = 0; k < CONV_Y / 4; ++k) {
        const int o = CONV_Y / 4 * w + k;
        double s = sm[o * 64 + lane];
        for (int j = 1; j < 4; ++j) s += sm[(j * CONV_Y + o) * 64 + lane];
        const int iy = y0 + CONV_Y * ly + o, ix = x0 + lx;
        if (iy < GY && ix < GX) conv_store<MODE>(out, Hs, iy, ix, iz, GY, GX, num, Y, X, s);
    }
}

// Any reach.  A thread per voxel, TY x 64 / TY of them along y and x a workgroup of one wavefront (TY: fitted to the grid's
// y side), which brings the columns along y that they reach into LDS (CONV_COLS at once, CONV_SEG voxels at a time), so
// a column is read and, for the adjoint, divided once for all of them.  Sums run over z, x, y ascending.  h: the
// (hr + 1)^3 weights of the cone's even octant.  Bound by a product's two loads, value and weight: 40 x 240 x 40 voxels at
// a reach of 14, 12,893 weights, forward 2.2 ms, adjoint 2.5, against 5.0 and 6.4 with every value read (and divided)
// from memory for each product; 32 x 4 x 32 voxels 0.41 and 0.46 ms against 1.9 and 2.1.
constexpr int CONV_SEG = 256, CONV_COLS = 4;
template <int MODE>
__global__ __launch_bounds__(64) void k_conv_any(const double *__restrict__ src, const double *__restrict__ Hs,
                                                 const double *__restrict__ h, const int32_t *__restrict__ lim, int hr, int GY,
                                                 int GX, int GZ, int num, int Y, int X, int TY, double *__restrict__ out) {
    __shared__ double col[CONV_COLS][CONV_SEG];
    const int t = threadIdx.x, TX = 64 / TY, W = hr + 1;
    const int tilesY = (GY + TY - 1) / TY, tilesX = (GX + TX - 1) / TX;
    const unsigned tile = blockIdx.x / tilesY;
    const int y0 = (int)(blockIdx.x % tilesY) * TY, x0 = (int)(tile % tilesX) * TX, iz = (int)(tile / tilesX);
    const int iy = y0 + t % TY, ix = x0 + t / TY;
    const int ya = max(y0 - hr, 0), yb = min(y0 + TY + hr, GY), xa = max(x0 - hr, 0), xb = min(x0 + TX + hr, GX);
    const int64_t n3 = (int64_t)num * num * num;
    CvAxis az(max(iz - hr, 0), num, num * num, n3 * Y * X);
    double s = 0;
    for (int z = max(iz - hr, 0); z <= min(iz + hr, GZ - 1); ++z, az.next()) {
        const int dz = abs(z - iz);
        CvAxis ax(xa, num, num, n3 * Y);
        for (int xc = xa; xc < xb; xc += CONV_COLS) {
            int64_t off[CONV_COLS];
#pragma unroll
            for (int c = 0; c < CONV_COLS; ++c, ax.next()) off[c] = az.off + (xc + c < xb ? ax.off : 0);
            for (int ys = ya; ys < yb; ys += CONV_SEG) {
                const int len = min(CONV_SEG, yb - ys);
                for (int k = t; k < len; k += 64) {
                    const int64_t oy = CvAxis(ys + k, num, 1, n3).off;
                    double v[CONV_COLS];
#pragma unroll
                    for (int c = 0; c < CONV_COLS; ++c) v[c] = MODE == 2 ? 1.0 : src[off[c] + oy];
#pragma unroll
                    for (int c = 0; c < CONV_COLS; ++c) {
                        if (MODE == 1) v[c] /= Hs[ys + k + (int64_t)GY * ((xc + c < xb ? xc + c : 0) + (int64_t)GX * z)];
                        col[c][k] = v[c];
                    }
                }
                __syncthreads();
                for (int x = xc; x < min(xc + CONV_COLS, xb); ++x) {
                    const int dx = abs(x - ix), last = dx <= hr ? lim[dx + (int64_t)W * dz] : -1;
                    const double *hx = h + (int64_t)W * (min(dx, hr) + (int64_t)W * dz), *cx = col[x - xc];
                    const int d1 = min(last, ys + len - 1 - iy);
#pragma unroll 4
                    for (int d = max(-last, ys - iy); d <= d1; ++d) s += hx[abs(d)] * cx[iy + d - ys];
                }
                __syncthreads();
            }
        }
    }
    if (iy < GY && ix < GX) conv_store<MODE>(out, Hs, iy, ix, iz, GY, GX, num, Y, X, s);
}

// A cone of one voxel (reach 0): 1.7 million voxels 12.5 us, where the forms above take 26 to bring rows for a single product.
template <int MODE>
__global__ void k_conv_point(const double *__restrict__ src, const double *__restrict__ Hs, const double *__restrict__ h,
                             int GY, int GX, int GZ, int num, int Y, int X, double *__restrict__ out) {
    const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (int64_t)GY * GX * GZ) return;
    const int iy = (int)(p % GY), ix = (int)((p / GY) % GX), iz = (int)(p / ((int64_t)GY * GX));
    const double v = MODE == 2 ? 1.0 : src[cv_new_index(iy, ix, iz, num, Y, X)];
    conv_store<MODE>(out, Hs, iy, ix, iz, GY, GX, num, Y, X, h[0] * (MODE == 1 ? v / Hs[p] : v));
}

}  // namespace

// ---------------------------------------------------------------------------------------------
namespace {

static_assert(2 * sizeof(OcState) <= 16 * sizeof(double) && RED_BLOCKS <= 2 * (OC_NODES + 1) * OC_BLOCKS &&
                  (size_t)2 * (OC_NODES + 1) * OC_BLOCKS + 16 <= SCRATCH_DOUBLES,
              "the OC update's working memory");

// Sum, dot, maximum or sharpness of device arrays on st, to the host.
double reduce_dev(int op, const double *a, const double *b, int64_t n, hipStream_t st) {
    const char *id = "tg_reduce:Input";
    if (op != R_SUM && op != R_DOT && op != R_MAXABSDIFF && op != R_SHARP) fail(TG_ERR_ARGS, id, "unknown reduction %d", op);
    Scratch sc(st);
    double *part = sc.dbl();
    const unsigned long long seq = sc.next();
#define TG_RED_CASE(OP)                                                                                   \
    case OP:                                                                                              \
        k_red_partial<OP><<<RED_BLOCKS, RED_THREADS, 0, st>>>(a, b, n, part);                             \
        k_red_final<OP><<<1, RED_THREADS, 0, st>>>(part, RED_BLOCKS, sc.host(), sc.seq_ptr(), seq);       \
        break;
    switch (op) { TG_RED_CASE(R_SUM) TG_RED_CASE(R_DOT) TG_RED_CASE(R_MAXABSDIFF) TG_RED_CASE(R_SHARP) }
#undef TG_RED_CASE
    TG_LAUNCH_CHECK(id);
    return *sc.wait(id);
}

}  // namespace

Filter::Filter(const tg_model &mm, double rMin, hipStream_t s) : m(mm), st(s) {
    const char *id = "tg_filter_create:Input";
    const HostLevel &L = m.lv[0];
    g.EY = L.resY; g.EX = L.resX; g.EZ = L.resZ;
    g.NY = L.resY + 1; g.NX = L.resX + 1; g.NZ = L.resZ + 1;
    Ne = L.Ne;
    double K[64];
    pde_filter_kernel(rMin, 1.0, K);  // eleSize(1) = 1 on the finest level (TOP_GPU.m:2066)
    // a cube of the Laplacian and the mass: one entry per number of edges between two corners
    kd[0] = K[0];
    kd[1] = K[1];
    kd[2] = K[2];
    kd[3] = K[6];
    // the preconditioner 1 / (sum of the diagonal entries of the elements around a node), per set of elements
    double tab[256];
    for (int c = 0; c < 256; ++c) {
        double s = 0;
        for (int j = 0; j < 8; ++j)
            if (c & (1 << j)) s += K[9 * vtx_of(!(j & 1), !(j & 2), !(j & 4))];
        tab[c] = c ? 1.0 / s : 0.0;
    }
    inv.upload(tab, 256, st);
    eleFwd.upload(L.eleMapForward, st);
    std::vector<int32_t> ef(L.Ne);
    for (int64_t k = 0; k < L.Ne; ++k) ef[k] = L.eleMapBack[k] - 1;
    eleFull0.upload(ef, st);
    DevBuf<uint8_t> solid;
    solid.upload(L.solid, st);
    code.alloc(g.nodes());
    k_filter_codes<<<grid_for(g.nodes(), 256), 256, 0, st>>>(solid, g, code);
    TG_LAUNCH_CHECK(id);
    y.alloc(g.nodes());
    pw.init(g.nodes(), st);
    // the tile: the fewest workgroups a plane (rims included, a tile is at most FS_THREADS nodes)
    int64_t best = INT64_MAX;
    for (int n = (int)((g.NY + FS_THREADS / 3 - 3) / (FS_THREADS / 3 - 2)); n <= g.NY; ++n) {
        const int cy = (g.NY + n - 1) / n, cx = FS_THREADS / (cy + 2) - 2;
        const int64_t count = (int64_t)((g.NY + cy - 1) / cy) * ((g.NX + cx - 1) / cx);
        if (count < best) {
            best = count;
            ty = cy;
            tx = cx;
        }
        if (cy <= 16) break;  // shorter runs along y are not worth a few workgroups
    }
    tyn = (g.NY + ty - 1) / ty;
    tiles = (int)best;
    // The chunk: its planes are read once and the two beside it again; a plane takes a latency (as long as
    // one workgroup's share of the traffic) and the shares of the workgroups on the compute unit.
    int dev = 0, cus = 0;
    TG_HIP(hipGetDevice(&dev), id);
    TG_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), id);
    cus = std::max(cus, 1);
    best = INT64_MAX;
    for (int z = 1; z <= g.NZ; ++z) {
        const int64_t n = (int64_t)tiles * ((g.NZ + z - 1) / z), cost = (z + 2) * (1 + (n + cus - 1) / cus);
        if (cost < best) {
            best = cost;
            chunk = z;
        }
    }
    chunks = (g.NZ + chunk - 1) / chunk;
    np = (int)std::min<int64_t>(RED_BLOCKS, (g.nodes() + 2 * RED_THREADS - 1) / (2 * RED_THREADS));
    parts.alloc((int64_t)tiles * chunks + 2 * np);
    TG_HIP(hipStreamSynchronize(st), id);
}

void Filter::apply(const double *src, double *tar, double tol, int maxIT, int *its, double *res) {
    const char *id = "tg_filter_apply:Numeric";
    double *prr = parts, *pzr = prr + np, *ppv = pzr + np;
    k_e2n<<<np, E2N_THREADS, 0, st>>>(src, eleFwd, code, g, inv, pw.r, prr, pzr);
    const dim3 grid((unsigned)tiles, (unsigned)chunks);
    FilterStep a{g, ty, tx, tyn, chunk, kd[0], kd[1], kd[2], kd[3], code, inv, pw.r, pw.z, pw.p, y, pw.v,
                 prr, pzr, np, ppv, pw.scal, pw.d_hscal, 0, S_XB, S_XA};
    k_filter_step<0><<<grid, FS_THREADS, 0, st>>>(a);
    int it = 0;
    double rn = 0;
    for (it = 1; it <= maxIT; ++it) {
        k_filter_update<<<np, RED_THREADS, 0, st>>>(pw.r, pw.v, g.nodes(), code, inv, ppv, tiles * chunks, pw.scal,
                                                    a.xn, prr, pzr);
        std::swap(a.xn, a.xo);
        std::swap(a.p, a.pold);
        a.seq = ++pw.seq;
        if (it == 1) k_filter_step<1><<<grid, FS_THREADS, 0, st>>>(a);
        else k_filter_step<2><<<grid, FS_THREADS, 0, st>>>(a);
        TG_LAUNCH_CHECK(id);
        rn = std::sqrt(pw.wait_rr()) / std::sqrt(pw.h_scal[S_BB]);
        if (!std::isfinite(rn)) fail(TG_ERR_NUMERIC, id, "non-finite residual at iteration %d", it);
        if (rn < tol) break;
    }
    if (its) *its = std::min(it, maxIT);
    if (res) *res = rn;
    k_n2e<<<grid_for(Ne, 256), 256, 0, st>>>(y, eleFull0, Ne, g, tar);
    TG_LAUNCH_CHECK(id);
}

ConvFilter::ConvFilter(int nelx, int nely, int nelz, double r, int n, hipStream_t s) : num(n), st(s) {
    const char *id = "tg_convfilter_create:Input";
    X = nelx; Y = nely; Z = nelz;
    GY = num * nely; GX = num * nelx; GZ = num * nelz;
    hr = (int)std::ceil(r) - 1;
    const int w = hr + 1;
    // [dy,dx,dz] = meshgrid(-c+1:c-1, ...); h = max(0, r - sqrt(dx^2+dy^2+dz^2)) (TOP_GPU.m:116-118): even in
    // each direction, so one octant; and the last dy with a weight of every row
    std::vector<double> h((size_t)w * w * w);
    std::vector<int32_t> last((size_t)w * w, -1);
    for (int dz = 0; dz < w; ++dz)
        for (int dx = 0; dx < w; ++dx)
            for (int dy = 0; dy < w; ++dy) {
                const double v = std::max(0.0, r - std::sqrt((double)dx * dx + (double)dy * dy + (double)dz * dz));
                h[dy + (size_t)w * (dx + (size_t)w * dz)] = v;
                if (v > 0) last[dx + (size_t)w * dz] = dy;
            }
    hd.upload(h, st);
    lim.upload(last, st);
    const int64_t ng = (int64_t)GY * GX * GZ;
    Hs.alloc(ng);
    // lanes along y and x of a workgroup's plane: the least (products + staging) over the grid that fits the LDS
    LY = 0;
    double least = 1e300;
    for (int ly = 1; ly <= 16 && hr >= 1 && hr <= CONV_HR && GZ <= 65535; ++ly)
        for (int lanes = 64; lanes >= 32; lanes -= 16) {
            // a column stride of 1 mod 8 doubles: the lanes' reads then fall on different banks
            const int lx = lanes / ly, rows = CONV_Y * ly + 2 * hr, cols = lx + 2 * hr, pi = (rows + 6) / 8 * 8 + 1;
            if (4 * (size_t)cols * pi * sizeof(double) > 64 * 1024) continue;
            const double tiles = std::ceil(GY / (double)(CONV_Y * ly)) * std::ceil(GX / (double)lx);
            const double t = tiles * (0.5 * w * w * w * CONV_Y + 0.5 * w * ((rows + 63) / 64) * cols);
            if (t < least) {
                least = t;
                LY = ly;
                LX = lx;
                pitch = pi;
            }
        }
    convolve<2>(nullptr, Hs);
    TG_HIP(hipStreamSynchronize(st), id);
}

template <int MODE>
void ConvFilter::convolve(const double *src, double *out) {
    const size_t lds = std::max(4 * (size_t)(LX + 2 * hr) * pitch, (size_t)4 * CONV_Y * 64) * sizeof(double);
    const dim3 grid(grid_for(GY, CONV_Y * std::max(LY, 1)) * grid_for(GX, std::max(LX, 1)), (unsigned)GZ);
    switch (LY || hr == 0 ? hr : -1) {
#define TG_CONV_CASE(H) \
    case H: k_conv<H, MODE><<<grid, 256, lds, st>>>(src, Hs, hd, lim, GY, GX, GZ, num, Y, X, LY, LX, pitch, out); break;
        case 0: {
            const int64_t ng = (int64_t)GY * GX * GZ;
            k_conv_point<MODE><<<grid_for(ng, 256), 256, 0, st>>>(src, Hs, hd, GY, GX, GZ, num, Y, X, out);
            break;
        }
        TG_CONV_CASE(1) TG_CONV_CASE(2) TG_CONV_CASE(3) TG_CONV_CASE(4) TG_CONV_CASE(5) TG_CONV_CASE(6)
        TG_CONV_CASE(7) TG_CONV_CASE(8) TG_CONV_CASE(9) TG_CONV_CASE(10) TG_CONV_CASE(11) TG_CONV_CASE(12)
#undef TG_CONV_CASE
        default: {
            int ty = 64;
            while (ty > 1 && ty >= 2 * GY) ty /= 2;
            const unsigned tiles = grid_for(GY, ty) * grid_for(GX, 64 / ty) * (unsigned)GZ;
            k_conv_any<MODE><<<tiles, 64, 0, st>>>(src, Hs, hd, lim, hr, GY, GX, GZ, num, Y, X, ty, out);
        }
    }
    TG_LAUNCH_CHECK("tg_convfilter:convolve");
}

void ConvFilter::forward(const double *x, double *out) { convolve<0>(x, out); }
void ConvFilter::adjoint(const double *dc, double *out) { convolve<1>(dc, out); }

}  // namespace tg

using namespace tg;

extern "C" {

int tg_solver_unit_compliance(tg_solver *s, const double *d_U, double *d_ce) {
    return guard("tg_solver_unit_compliance:Input", [&] {
        const char *id = "tg_solver_unit_compliance:Input";
        if (!s || !s->s || !d_U || !d_ce) fail(TG_ERR_ARGS, id, "null argument");
        Solver &S = *s->s;
        DevLevel &F = S.lv[0];
        k_unpack<double, double><<<grid_for(F.g.nodes(), 256), 256, 0, S.st>>>(d_U, S.pw.z, F.nodFwd, F.g.nodes());
        if (S.super) {
            if (!S.assembled) fail(TG_ERR_STATE, "tg_solver_unit_compliance:State", "assemble first (K_mat)");
            k_unit_compliance_super<<<grid_for(F.Ne, UC_ELEMS), UC_PARTS * UC_ELEMS, 0, S.st>>>(S.pw.z, F.Ks64, F.ldk, F.eleFull0, F.Ne, F.g, d_ce);
        } else {
            k_unit_compliance<<<grid_for(F.Ne, 256), 256, 0, S.st>>>(S.pw.z, S.K0_64, F.eleFull0, F.Ne, F.g, d_ce);
        }
        TG_LAUNCH_CHECK(id);
        TG_HIP(hipStreamSynchronize(S.st), id);
    });
}

int tg_compliance_grad(tg_solver *s, tg_filter *f, const double *d_x, double Emin, double E0, double penal,
                       double tol, int32_t max_it, double filter_tol, int32_t warm, double *d_U, double *c_out,
                       double *d_dcdx, int32_t *its_out) {
    return guard("tg_compliance_grad:Input", [&] {
        const char *id = "tg_compliance_grad:Input";
        if (!s || !s->s || !d_x || !d_U || !c_out || max_it < 1) fail(TG_ERR_ARGS, id, "bad arguments");
        Solver &S = *s->s;
        if (S.super) fail(TG_ERR_STATE, "tg_compliance_grad:State", "standard voxel mode only");
        if (f && (!f->f || f->f->Ne != S.lv[0].Ne)) fail(TG_ERR_ARGS, id, "filter does not match the solver's mesh");
        const hipStream_t st = S.st;
        const int64_t Ne = S.lv[0].Ne, ndof = 3 * S.lv[0].Nn;
        if ((int64_t)S.adjF.n != ndof) {
            S.adjF.upload(S.model.F.data(), ndof, st);  // load case 1
            S.adjXp.alloc(Ne);
            S.adjE.alloc(Ne);
            S.adjCe.alloc(Ne);
            S.adjG.alloc(Ne);
        }
        int fits = 0;
        double fres = 0;
        // xPhys = filter(x)
        if (f) {
            TG_HIP(hipStreamSynchronize(st), id);
            f->f->apply(d_x, S.adjXp, filter_tol, max_it, &fits, &fres);
            TG_HIP(hipStreamSynchronize(f->f->st), id);
        } else {
            TG_HIP(hipMemcpyAsync(S.adjXp.p, d_x, Ne * sizeof(double), hipMemcpyDeviceToDevice, st), id);
        }
        // E, K(E) U = F
        k_simp<<<grid_for(Ne, 256), 256, 0, st>>>(S.adjXp, S.adjE, Ne, Emin, E0, penal);
        TG_LAUNCH_CHECK(id);
        S.set_modulus(S.adjE);
        S.assemble();
        int its = 0;
        double res = 0;
        S.pcg(S.adjF, d_U, tol, max_it, warm, &its, &res);
        // ce_e = u_e' K0 u_e, c = sum E_e ce_e, g = -p (E0 - Emin) xPhys^(p-1) ce
        DevLevel &F = S.lv[0];
        k_unpack<double, double><<<grid_for(F.g.nodes(), 256), 256, 0, st>>>(d_U, S.pw.z, F.nodFwd, F.g.nodes());
        k_unit_compliance<<<grid_for(Ne, 256), 256, 0, st>>>(S.pw.z, S.K0_64, F.eleFull0, Ne, F.g, S.adjCe);
        TG_LAUNCH_CHECK(id);
        *c_out = reduce_dev(R_DOT, S.adjE, S.adjCe, Ne, st);
        if (d_dcdx) {
            k_sens<<<grid_for(Ne, 256), 256, 0, st>>>(S.adjXp, S.adjCe, f ? S.adjG.p : d_dcdx, Ne, 1, Emin, E0, penal, 1.0);
            TG_LAUNCH_CHECK(id);
            if (f) {  // the Helmholtz filter is symmetric: its adjoint is the forward filter
                TG_HIP(hipStreamSynchronize(st), id);
                f->f->apply(S.adjG, d_dcdx, filter_tol, max_it, &fits, &fres);
                TG_HIP(hipStreamSynchronize(f->f->st), id);
            }
        }
        TG_HIP(hipStreamSynchronize(st), id);
        if (its_out) *its_out = its;
    });
}

int tg_solver_subvoxel_energy(tg_solver *s, const double *d_U, double *d_dc) {
    return guard("tg_solver_subvoxel_energy:Input", [&] {
        const char *id = "tg_solver_subvoxel_energy:Input";
        if (!s || !s->s || !d_U || !d_dc) fail(TG_ERR_ARGS, id, "null argument");
        Solver &S = *s->s;
        if (!S.super) fail(TG_ERR_STATE, id, "super-element mode only");
        DevLevel &F = S.lv[0];
        k_unpack<double, double><<<grid_for(F.g.nodes(), 256), 256, 0, S.st>>>(d_U, S.pw.z, F.nodFwd, F.g.nodes());
        k_subvoxel_energy<<<grid_for(F.Ne, 16), 256, 0, S.st>>>(S.pw.z, S.Imat, F.eleFull0, F.Ne, F.g, d_dc);
        TG_LAUNCH_CHECK(id);
        TG_HIP(hipStreamSynchronize(S.st), id);
    });
}

int tg_simp_modulus(const double *d_x, int64_t n, double Emin, double E0, double penal, double *d_E, void *stream) {
    return guard("tg_simp_modulus:Input", [&] {
        if (!d_x || !d_E || n < 0) fail(TG_ERR_ARGS, "tg_simp_modulus:Input", "bad arguments");
        if (n) k_simp<<<grid_for(n, 256), 256, 0, (hipStream_t)stream>>>(d_x, d_E, n, Emin, E0, penal);
        TG_LAUNCH_CHECK("tg_simp_modulus:HIP");
    });
}

int tg_sensitivity(const double *d_x, const double *d_ce, int64_t n, int32_t per, double Emin, double E0, double penal,
                   double cSolid, double *d_dc, void *stream) {
    return guard("tg_sensitivity:Input", [&] {
        if (!d_x || !d_ce || !d_dc || n < 0 || per < 1) fail(TG_ERR_ARGS, "tg_sensitivity:Input", "bad arguments");
        if (n) k_sens<<<grid_for(n, 256), 256, 0, (hipStream_t)stream>>>(d_x, d_ce, d_dc, n, per, Emin, E0, penal, cSolid);
        TG_LAUNCH_CHECK("tg_sensitivity:HIP");
    });
}

int tg_elementwise(int32_t op, const double *d_a, const double *d_b, double scalar, int64_t n, double *d_out,
                   void *stream) {
    return guard("tg_elementwise:Input", [&] {
        if (!d_a || !d_b || !d_out || n < 0) fail(TG_ERR_ARGS, "tg_elementwise:Input", "bad arguments");
        hipStream_t st = (hipStream_t)stream;
        if (!n) return;
        if (op == TG_EW_MUL) k_mul<<<grid_for(n, 256), 256, 0, st>>>(d_a, d_b, d_out, n);
        else if (op == TG_EW_DIV_FLOOR) k_div_floor<<<grid_for(n, 256), 256, 0, st>>>(d_a, d_b, d_out, scalar, n);
        else if (op == TG_EW_SET_WHERE) k_set_where<<<grid_for(n, 256), 256, 0, st>>>(d_a, d_b, d_out, scalar, n);
        else if (op == TG_EW_AXPY) k_axpy<<<grid_for(n, 256), 256, 0, st>>>(d_a, d_b, d_out, scalar, n);
        else fail(TG_ERR_ARGS, "tg_elementwise:Input", "unknown op %d", op);
        TG_LAUNCH_CHECK("tg_elementwise:HIP");
    });
}

int tg_reduce(int32_t op, const double *d_a, const double *d_b, int64_t n, double *out, void *stream) {
    return guard("tg_reduce:Input", [&] {
        if (!d_a || !out || n < 0 || ((op == TG_RED_DOT || op == TG_RED_MAXABSDIFF) && !d_b))
            fail(TG_ERR_ARGS, "tg_reduce:Input", "bad arguments");
        *out = reduce_dev(op, d_a, d_b, n, (hipStream_t)stream);
    });
}

int tg_oc_update(const double *d_x, const double *d_dc, const double *d_dv, const double *d_passive, int64_t n,
                 double fval, double move, double *d_xnew, double *change, int32_t *bisections, void *stream) {
    return guard("tg_oc_update:Input", [&] {
        const char *id = "tg_oc_update:Input";
        if (!d_x || !d_dc || !d_dv || !d_xnew || n < 1) fail(TG_ERR_ARGS, id, "bad arguments");
        hipStream_t st = (hipStream_t)stream;
        const int nb = (int)std::min<int64_t>(OC_BLOCKS, (n + RED_THREADS - 1) / RED_THREADS);
        auto apart = [&](const double *a) { return !a || a + n <= d_xnew || d_xnew + n <= a; };
        double *b = apart(d_x) && apart(d_dc) && apart(d_dv) && apart(d_passive) ? d_xnew : nullptr;
        Scratch sc(st);
        // 16 doubles of states, then the sums of two launches, whose place the maxima take after the last one
        OcState *state = (OcState *)sc.dbl();
        double *part[2] = {sc.dbl() + 16, sc.dbl() + 16 + (size_t)(OC_NODES + 1) * nb}, *maxima = part[0];
        int k = 0;  // launches; launch k's sums are in part[k & 1], and it left the state before them in state[k & 1]
        OcState s{0.0, 1e9, 0.0, 0.0, 0.0};
        // (l2-l1)/(l1+l2) halves each step from 1: at most ~100 steps, more than 48 but for the largest
        // multipliers; check after 48, then every 16
        for (int upto = 48; ; upto += 16) {
            for (; OC_DEPTH * k < upto; ++k) {
                const OcState *old = state + ((k + 1) & 1);
                const double *in = part[(k + 1) & 1];
                if (k == 0)
                    k_oc_pass<0><<<nb, RED_THREADS, 0, st>>>(d_x, d_dc, d_dv, b, d_passive, n, fval, move, nullptr, state,
                                                             nullptr, part[0]);
                else if (k == 1)
                    k_oc_pass<1><<<nb, RED_THREADS, 0, st>>>(d_x, d_dc, d_dv, b, d_passive, n, fval, move, old, state + 1, in,
                                                             part[1]);
                else
                    k_oc_pass<2><<<nb, RED_THREADS, 0, st>>>(d_x, d_dc, d_dv, b, d_passive, n, fval, move, old,
                                                             state + (k & 1), in, part[k & 1]);
            }
            const unsigned long long seq = sc.next();
            k_oc_close<<<1, RED_THREADS, 0, st>>>(n, fval, state + ((k - 1) & 1), state + (k & 1), part[(k - 1) & 1], nb,
                                                  sc.host(), sc.seq_ptr(), seq);
            TG_LAUNCH_CHECK(id);
            std::memcpy(&s, sc.wait(id), sizeof s);
            if (!((s.l2 - s.l1) / (s.l1 + s.l2) > 1e-6)) break;
            if (upto > 400) fail(TG_ERR_NUMERIC, "tg_oc_update:Numeric", "bisection did not converge");
        }
        const unsigned long long seq = sc.next();
        k_oc_apply<<<RED_BLOCKS, RED_THREADS, 0, st>>>(d_x, d_dc, d_dv, d_passive, d_xnew, n, move, state + (k & 1), maxima);
        k_red_final<R_MAXABSDIFF><<<1, RED_THREADS, 0, st>>>(maxima, RED_BLOCKS, sc.host(), sc.seq_ptr(), seq);
        TG_LAUNCH_CHECK(id);
        const double m = *sc.wait(id);
        if (change) *change = m;
        if (bisections) *bisections = 16 * (int)std::ceil(s.steps / 16);
    });
}

int tg_filter_create(const tg_model *m, double rMin, void *stream, tg_filter **out) {
    return guard("tg_filter_create:Input", [&] {
        if (!m || !out) fail(TG_ERR_ARGS, "tg_filter_create:Input", "null argument");
        auto *f = new tg_filter();
        try {
            f->f = new Filter(*m, rMin, (hipStream_t)stream);
        } catch (...) {
            delete f;
            throw;
        }
        *out = f;
    });
}

void tg_filter_destroy(tg_filter *f) {
    if (!f) return;
    if (f->f) (void)hipStreamSynchronize(f->f->st);
    delete f->f;
    delete f;
}

int tg_filter_apply(tg_filter *f, const double *d_src, double *d_tar, double tol, int32_t max_it, int32_t *its) {
    return guard("tg_filter_apply:Input", [&] {
        if (!f || !f->f || !d_src || !d_tar || max_it < 1) fail(TG_ERR_ARGS, "tg_filter_apply:Input", "bad arguments");
        int it = 0;
        double res = 0;
        f->f->apply(d_src, d_tar, tol, max_it, &it, &res);
        TG_HIP(hipStreamSynchronize(f->f->st), "tg_filter_apply:HIP");
        if (its) *its = it;
    });
}

int tg_convfilter_create(int32_t nelx, int32_t nely, int32_t nelz, double rMin_subvoxels, int32_t num, void *stream,
                         tg_convfilter **out) {
    return guard("tg_convfilter_create:Input", [&] {
        if (!out || nelx < 1 || nely < 1 || nelz < 1 || num < 1 || !(rMin_subvoxels > 0))
            fail(TG_ERR_ARGS, "tg_convfilter_create:Input", "bad arguments");
        auto *f = new tg_convfilter();
        try {
            f->f = new ConvFilter(nelx, nely, nelz, rMin_subvoxels, num, (hipStream_t)stream);
        } catch (...) {
            delete f;
            throw;
        }
        *out = f;
    });
}

void tg_convfilter_destroy(tg_convfilter *f) {
    if (!f) return;
    if (f->f) (void)hipStreamSynchronize(f->f->st);
    delete f->f;
    delete f;
}

int tg_convfilter_forward(tg_convfilter *f, const double *d_x, double *d_out) {
    return guard("tg_convfilter_forward:Input", [&] {
        if (!f || !f->f || !d_x || !d_out) fail(TG_ERR_ARGS, "tg_convfilter_forward:Input", "null argument");
        f->f->forward(d_x, d_out);
    });
}

int tg_convfilter_adjoint(tg_convfilter *f, const double *d_dc, double *d_out) {
    return guard("tg_convfilter_adjoint:Input", [&] {
        if (!f || !f->f || !d_dc || !d_out) fail(TG_ERR_ARGS, "tg_convfilter_adjoint:Input", "null argument");
        f->f->adjoint(d_dc, d_out);
    });
}

}  // extern "C"
