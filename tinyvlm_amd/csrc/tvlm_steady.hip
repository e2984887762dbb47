// tvlm_steady.hip -- steady VLM solves of a batch of requests (the caller of the hot path,
// VLM::run, vlm/src/vlm.cpp:97-151, for many angles of attack at once).
//
// A plan owns the device buffers of `batch` requests on one mesh (any number of surfaces).  For
// request b, solve() repeats VLM::run's sequence: wing reset to the input mesh, wake row shed,
// displacement 100 chords along -freestream, second shed, panel metrics at alpha_b, influence matrix
// (iteration 1: the trailing-edge columns also see the one wake row), rhs = -(V_inf . n), solve,
// circulation differences, steady forces and per-surface CL/CM.
//   mode 0 (plain FP64): exact FP64 assembly, FP64 LU and substitution, one request after another;
//                        the reference's terms, IEEE square roots and divisions and cutoffs, with the
//                        segments shared between rings and contracted (SegForm).
//   mode 1 (served)    : every request's FP64 influence matrix in the seeded form, stored rounded to
//                        FP32 as well, one batched FP32 LU for all requests, then FP64 iterative refinement
//                        x += A32^{-1} (b - A64 x) (kRefine + 1 corrections, residual in FP64 against
//                        the FP64 matrix), so the answer carries the FP64 matrix's accuracy.  The
//                        returned x of every request is checked: ||b - A64 x||_inf <= sqrt(N) eps
//                        ||x||_inf ||A64||_inf (the stopping test of LAPACK's dsgesv).  A request that
//                        fails it gets more corrections (up to kMaxCorrections in all), then, if it
//                        still fails, the FP64 LU of its FP64 matrix (the plain path's solve); a request
//                        whose FP32 LU had a cooperative panel give up waiting (info -999) is first
//                        re-factored with one-group panels.  tvlm_vlm_refinement reports what each
//                        request took.
// Per-surface coefficients are combined on the host (area-weighted CL, area*MAC-weighted CM,
// vlm/src/vlm_backend.cpp:71-139).
#include <cmath>
#include <cstring>
#include <vector>

#include "tvlm_internal.hpp"

namespace {
constexpr int kMaxS = TVLM_MAX_SURFACES;
constexpr int kRefine = 3;
constexpr int kMaxCorrections = 8;  // corrections of one request before the FP64 fallback
// tvlm_vlm_refinement status bits
constexpr int32_t kStMoreCorrections = 1, kStFallback64 = 2, kStRefactored = 4, kStUnresolved = 8;
constexpr int kResidRows = 64;     // rows per work-group of the residual
constexpr int kResidWaves = 8;     // waves splitting its columns
}  // namespace

struct tvlm_vlm_plan {
    int32_t mode = 0, n_surf = 0, N = 0, batch = 0, active = 0;
    hipStream_t stream = nullptr;
    int64_t ns[kMaxS] = {}, nc[kMaxS] = {}, off[kMaxS] = {};  // off: first panel of surface m
    int64_t vsz[kMaxS] = {}, wsz[kMaxS] = {}, psz[kMaxS] = {};  // elements per request: verts, wake, panels
    std::vector<void*> allocs;
    int64_t bytes = 0;                                           // device bytes held
    hipEvent_t done = nullptr;  // recorded after the plan's own latest work (creation, solve, results)
    double* init[kMaxS] = {};                                    // {ns+1, nc+1, 4}
    double *verts[kMaxS] = {}, *wake[kMaxS] = {};                // per request b: + b * vsz / wsz
    double *colloc[kMaxS] = {}, *normals[kMaxS] = {}, *areas[kMaxS] = {};
    double *vel[kMaxS] = {}, *forces[kMaxS] = {}, *gdelta[kMaxS] = {};
    double *lhs = nullptr, *rhs = nullptr, *x = nullptr, *res = nullptr, *coef = nullptr;
    double* par = nullptr;  // per request: 16 n_surf transform values, then kPar values (tvlm_vlm_solve_n)
    float *lhs32 = nullptr, *r32 = nullptr;
    int32_t *ipiv = nullptr, *info = nullptr;
    void* prep = nullptr;  // served mode: what getrs derives from the factors, once for all corrections
    double *rowabs = nullptr, *berr = nullptr;  // served mode: row sums of |A64|, backward error per request
    int32_t* conv = nullptr;                     // served mode: 1 = the request's x passed the test
    std::vector<int32_t> st_status, st_corr;     // per request of the last solve (tvlm_vlm_refinement)
    std::vector<double> st_berr;
    bool checked = false;                        // the last solve's requests were checked (and rescued)
    double* par_host = nullptr;  // pinned copy of par
    bool solved = false;
    tvlm_lhs_group* group = nullptr;  // served mode: every request's influence matrix, one grouped launch

    int alloc(void** p, size_t bytes) {
        TVLM_HIP(hipMalloc(p, bytes));
        allocs.push_back(*p);
        this->bytes += (int64_t)bytes;
        return TVLM_OK;
    }
};

namespace tvlm {
namespace {

constexpr int kPar = 12;  // alpha, freestream (3), lift axis (3), CM reference point (3), dynamic pressure

struct VSurf {
    const double* init;
    double *verts, *wake, *colloc, *normals, *areas, *vel, *forces, *gdelta;
    int64_t vsz, wsz, psz;  // elements per request: vertices, wake, panels
    int32_t ns, nc, off;
};

struct VTab {
    int32_t n, N, items;  // items: vertices and panels of all surfaces
    const double* par;
    double *rhs, *coef;
    const double* x;
    VSurf s[kMaxS];
};

// Geometry and rhs of requests b0 + blockIdx.y (vlm.cpp:97-124): a thread per vertex (the wing moved by
// the request's transform; its trailing edge before and after is the wake's one ring row) or per
// panel (metrics at alpha, freestream velocity, rhs = -(V . n)).
// Bound by the launches, so one for all requests: with a dozen small launches per request before and nine
// after its solve, 32 requests of 256 panels took 2.33 ms, with this kernel and k_vlm_post 0.77 ms.
__global__ __launch_bounds__(256) void k_vlm_geom(VTab t, int b0) {
    const int b = b0 + blockIdx.y;
    int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= t.items) return;
    int m = 0;
    for (; m + 1 < t.n; m++) {
        const int here = (t.s[m].ns + 1) * (t.s[m].nc + 1) + t.s[m].ns * t.s[m].nc;
        if (e < here) break;
        e -= here;
    }
    const VSurf& S = t.s[m];
    const double* par = t.par + (int64_t)b * (16 * t.n + kPar);
    const double* M = par + 16 * m;
    par += 16 * t.n;
    const int ns = S.ns, nc = S.nc, vs1 = ns + 1, nv = vs1 * (nc + 1), np = ns * nc;
    auto moved = [&](int v, int r) {
        const double x[4] = {S.init[v], S.init[v + nv], S.init[v + 2 * nv], S.init[v + 3 * nv]};
        return displace_row(M, 1, 4, r, x);
    };
    if (e < nv) {
        double* V = S.verts + b * S.vsz;
        double* W = S.wake + b * S.wsz;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const double y = moved(e, r);
            V[e + r * nv] = y;
            if (e / vs1 == nc) {
                W[e % vs1 + r * 2 * vs1] = y;
                W[vs1 + e % vs1 + r * 2 * vs1] = S.init[e + r * nv];
            }
        }
        return;
    }
    const int p = e - nv, i = p % ns, j = p / ns;
    auto vertex = [&](int v) -> v3<double> { return {moved(v, 0), moved(v, 1), moved(v, 2)}; };
    const int v0 = i + j * vs1;
    v3<double> c, n;
    double area;
    panel_metrics(par[0], vertex(v0), vertex(v0 + 1), vertex(v0 + 1 + vs1), vertex(v0 + vs1), c, n, area);
    const double fx = par[1], fy = par[2], fz = par[3];
    const int64_t o = b * S.psz;
    double *C = S.colloc + 3 * o, *Nn = S.normals + 3 * o, *U = S.vel + 3 * o;
    C[p] = c.x;
    C[p + np] = c.y;
    C[p + 2 * np] = c.z;
    Nn[p] = n.x;
    Nn[p + np] = n.y;
    Nn[p + 2 * np] = n.z;
    U[p] = fx;
    U[p + np] = fy;
    U[p + 2 * np] = fz;
    S.areas[o + p] = area;
    t.rhs[(int64_t)b * t.N + S.off + p] = -(fx * n.x + fy * n.y + fz * n.z);
}

constexpr int kVPostThreads = 1024;

// Circulation differences, steady forces and the coefficient sums of request b0 + blockIdx.x, one
// work-group (vlm.cpp:126-151): coef[(b n + m) * 8 + {0: area, 1: mac, 2: cl, 3..5: cm}], area and MAC
// only as such (CL and CM are formed from the surfaces' sums on the host).
__global__ __launch_bounds__(kVPostThreads) void k_vlm_post(VTab t, int b0) {
    __shared__ double red[kVPostThreads / 64][6];
    const int b = b0 + blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const double* par = t.par + (int64_t)b * (16 * t.n + kPar) + 16 * t.n;
    const v3<double> U = {par[1], par[2], par[3]}, la = {par[4], par[5], par[6]}, ref = {par[7], par[8], par[9]};
    for (int m = 0; m < t.n; m++) {
        const VSurf& S = t.s[m];
        const int ns = S.ns, nc = S.nc, vs1 = ns + 1, nv = vs1 * (nc + 1), np = ns * nc;
        const int64_t o = b * S.psz;
        const double* g = t.x + (int64_t)b * t.N + S.off;
        const double* V = S.verts + b * S.vsz;
        auto vertex = [&](int v) -> v3<double> { return {V[v], V[v + nv], V[v + 2 * nv]}; };
        double v[6] = {};
        for (int p = threadIdx.x; p < np; p += kVPostThreads) {
            const int i = p % ns, j = p / ns, va = i + j * vs1;
            const v3<double> a = vertex(va), e = vertex(va + 1);
            const double area = S.areas[o + p];
            const double gd = p >= ns ? g[p] - g[p - ns] : g[p];
            const v3<double> F = gd * cross(U, e - a);  // rho = 1 as in the reference (vlm_backend_cpu.cpp:282)
            S.gdelta[o + p] = gd;
            double* f = S.forces + 3 * o + p;
            f[0] = F.x;
            f[np] = F.y;
            f[2 * np] = F.z;
            const v3<double> lever = 0.5 * (a + e) - ref, mo = cross(lever, F);
            v[0] += area;
            v[2] += dot(F, la);
            v[3] += mo.x;
            v[4] += mo.y;
            v[5] += mo.z;
        }
        for (int i = threadIdx.x; i < ns; i += kVPostThreads) {
            const v3<double> l0 = vertex(i), l1 = vertex(i + 1);
            const v3<double> d0 = l0 - vertex(i + nc * vs1), d1 = l1 - vertex(i + 1 + nc * vs1), d3 = l1 - l0;
            const double c0 = sqrt(dot(d0, d0)), c1 = sqrt(dot(d1, d1));
            v[1] += 0.5 * (c0 * c0 + c1 * c1) * sqrt(dot(d3, d3));
        }
#pragma unroll
        for (int k = 0; k < 6; k++)
#pragma unroll
            for (int h = 32; h > 0; h >>= 1) v[k] += __shfl_xor(v[k], h, 64);
        __syncthreads();  // the previous surface's sums are read
        if (lane == 0)
            for (int k = 0; k < 6; k++) red[wave][k] = v[k];
        __syncthreads();
        if (threadIdx.x < 6) {
            const int k = threadIdx.x;
            double sum = 0.0, area = 0.0;
            for (int w = 0; w < kVPostThreads / 64; w++) {
                sum += red[w][k];
                area += red[w][0];
            }
            t.coef[((int64_t)b * t.n + m) * 8 + k] = k == 0 ? sum : k == 1 ? sum / area : sum / par[10];
        }
    }
}

// r = rhs - A x per request (FP64).  A work-group takes 64 rows (one per lane) and its 8 waves
// split the columns (wave w: columns w, w + 8, ...), so each wave reads 64 consecutive rows of a
// column (512 contiguous bytes) and N / 8 work-groups' worth of waves keep enough loads in flight
// to stream the FP64 matrix at HBM rate; x[j] is the same for the whole wave; the 8 partial sums
// are added in LDS in a fixed order.
// With ROWABS the same pass also stores the row sums of |A| (for ||A||_inf of the convergence test).
template <bool ROWABS>
__global__ __launch_bounds__(kResidRows * kResidWaves) void k_residual(const double* __restrict__ A, int n,
                                                                      const double* __restrict__ rhs,
                                                                      const double* __restrict__ x,
                                                                      double* __restrict__ r,
                                                                      double* __restrict__ rowabs) {
    __shared__ double part[kResidWaves][kResidRows];
    __shared__ double apart[ROWABS ? kResidWaves : 1][kResidRows];
    const int64_t b = blockIdx.y;
    A += b * (int64_t)n * n;
    rhs += b * n;
    x += b * n;
    r += b * n;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i = blockIdx.x * kResidRows + lane;
    double acc = 0.0, aacc = 0.0;
    if (i < n) {
        const double* Ai = A + i;
#pragma unroll 4
        for (int j = w; j < n; j += kResidWaves) {
            const double aij = Ai[(int64_t)j * n];
            acc += aij * x[j];
            if constexpr (ROWABS) aacc += fabs(aij);
        }
    }
    part[w][lane] = acc;
    if constexpr (ROWABS) apart[w][lane] = aacc;
    __syncthreads();
    if (w == 0 && i < n) {
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < kResidWaves; q++) s += part[q][lane];
        r[i] = rhs[i] - s;
        if constexpr (ROWABS) {
            double sa = 0.0;
#pragma unroll
            for (int q = 0; q < kResidWaves; q++) sa += apart[q][lane];
            rowabs[b * n + i] = sa;
        }
    }
}

// Convergence test of request blockIdx.x (LAPACK dsgesv's stopping test): with rnrm = ||r||_inf,
// xnrm = ||x||_inf, anrm = ||A||_inf (max row sum), converged iff the FP32 LU reported no problem
// (info == 0), every entry of r and x is finite and rnrm <= sqrt(n) eps xnrm anrm.  berr = rnrm /
// (xnrm anrm), the normwise backward error.
__global__ __launch_bounds__(256) void k_refine_check(const double* __restrict__ r, const double* __restrict__ x,
                                                      const double* __restrict__ rowabs,
                                                      const int32_t* __restrict__ info, int n,
                                                      double* __restrict__ berr, int32_t* __restrict__ conv) {
    __shared__ double sr[256], sx[256], sa[256];
    __shared__ int sbad[256];
    const int64_t b = blockIdx.x;
    r += b * n;
    x += b * n;
    rowabs += b * n;
    double mr = 0.0, mx = 0.0, ma = 0.0;
    int bad = 0;
    for (int i = threadIdx.x; i < n; i += 256) {
        const double ri = r[i], xi = x[i];
        bad |= !isfinite(ri) || !isfinite(xi);
        mr = fmax(mr, fabs(ri));
        mx = fmax(mx, fabs(xi));
        ma = fmax(ma, rowabs[i]);
    }
    sr[threadIdx.x] = mr;
    sx[threadIdx.x] = mx;
    sa[threadIdx.x] = ma;
    sbad[threadIdx.x] = bad;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (threadIdx.x < h) {
            sr[threadIdx.x] = fmax(sr[threadIdx.x], sr[threadIdx.x + h]);
            sx[threadIdx.x] = fmax(sx[threadIdx.x], sx[threadIdx.x + h]);
            sa[threadIdx.x] = fmax(sa[threadIdx.x], sa[threadIdx.x + h]);
            sbad[threadIdx.x] |= sbad[threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double rn = sr[0], xa = sx[0] * sa[0];
        const bool ok = info[b] == 0 && sbad[0] == 0 && rn <= sqrt((double)n) * 2.220446049250313e-16 * xa;
        berr[b] = sbad[0] ? (double)NAN : (xa > 0.0 ? rn / xa : (rn == 0.0 ? 0.0 : (double)INFINITY));
        conv[b] = ok ? 1 : 0;
    }
}

__global__ void k_to_f32(const double* __restrict__ src, float* __restrict__ dst, int64_t count) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = (float)src[i];
}

__global__ void k_add_f32(double* __restrict__ x, const float* __restrict__ d, int64_t count) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        x[i] += (double)d[i];
}

int grid_for(int64_t n) { return (int)((n + 255) / 256 < 4096 ? (n + 255) / 256 : 4096); }

void views(tvlm_vlm_plan* P, int b, int m, tvlm_view& v, tvlm_view& w, tvlm_view& c, tvlm_view& nn, tvlm_view& a,
           tvlm_view& vel, tvlm_view& f, tvlm_view& gd) {
    const int64_t ns = P->ns[m], nc = P->nc[m];
    v = {P->verts[m] + b * P->vsz[m], {ns + 1, nc + 1, 4}, {1, ns + 1, (ns + 1) * (nc + 1)}};
    w = {P->wake[m] + b * P->wsz[m], {ns + 1, 2, 4}, {1, ns + 1, (ns + 1) * 2}};
    c = {P->colloc[m] + b * 3 * P->psz[m], {ns, nc, 3}, {1, ns, ns * nc}};
    nn = {P->normals[m] + b * 3 * P->psz[m], {ns, nc, 3}, {1, ns, ns * nc}};
    a = {P->areas[m] + b * P->psz[m], {ns, nc, 1}, {1, ns, ns * nc}};
    vel = {P->vel[m] + b * 3 * P->psz[m], {ns, nc, 3}, {1, ns, ns * nc}};
    f = {P->forces[m] + b * 3 * P->psz[m], {ns, nc, 3}, {1, ns, ns * nc}};
    gd = {P->gdelta[m] + b * P->psz[m], {ns, nc, 1}, {1, ns, ns * nc}};
}

VTab table(const tvlm_vlm_plan* P) {
    VTab t{};
    t.n = P->n_surf;
    t.N = P->N;
    t.par = P->par;
    t.rhs = P->rhs;
    t.coef = P->coef;
    t.x = P->x;
    for (int m = 0; m < t.n; m++) {
        t.s[m] = {P->init[m], P->verts[m], P->wake[m], P->colloc[m], P->normals[m], P->areas[m], P->vel[m],
                  P->forces[m], P->gdelta[m], P->vsz[m], P->wsz[m], P->psz[m], (int32_t)P->ns[m], (int32_t)P->nc[m],
                  (int32_t)P->off[m]};
        t.items += (int32_t)(P->vsz[m] / 4 + P->psz[m]);
    }
    return t;
}

// geometry and rhs of requests [b0, b0 + count)
int geometry(tvlm_vlm_plan* P, int b0, int count) {
    const VTab t = table(P);
    hipLaunchKernelGGL(k_vlm_geom, dim3((t.items + 255) / 256, count), dim3(256), 0, P->stream, t, b0);
    TVLM_LAUNCHED();
    return TVLM_OK;
}

// circulation differences, forces and coefficients of requests [b0, b0 + count)
int post(tvlm_vlm_plan* P, int b0, int count) {
    hipLaunchKernelGGL(k_vlm_post, dim3(count), dim3(kVPostThreads), 0, P->stream, table(P), b0);
    TVLM_LAUNCHED();
    return TVLM_OK;
}

// influence matrix of request b, whose geometry stands (seeded: the served form)
int matrix(tvlm_vlm_plan* P, int b, bool seeded) {
    hipStream_t st = P->stream;
    const int n = P->n_surf;
    std::vector<tvlm_view> V(n), W(n), C(n), Nn(n), A(n), VEL(n), F(n), GD(n);
    for (int m = 0; m < n; m++) views(P, b, m, V[m], W[m], C[m], Nn[m], A[m], VEL[m], F[m], GD[m]);
    const int64_t NN = (int64_t)P->N * P->N;
    double* lhs = P->lhs + (P->mode == 1 ? b * NN : 0);
    TVLM_TRY(tvlm_fill_f64(0, lhs, 1, 0.0, NN, st));
    tvlm_view L = {lhs, {P->N, P->N, 1}, {1, P->N, NN}};
    if (seeded) return lhs_assemble_seeded_f64(&L, n, C.data(), Nn.data(), V.data(), W.data(), 1, st);
    return tvlm_lhs_assemble_f64(&L, n, C.data(), Nn.data(), V.data(), W.data(), 1, 0.0, st);
}

// Served mode, after the solve: reads the per-request test results; for every request that failed,
// (1) if its FP32 LU stalled (info -999), re-factors its FP32 copy with one-group panels and restarts
// its refinement from x = 0; (2) applies more corrections, one at a time with the test after each,
// up to kMaxCorrections in all; (3) if it still fails, solves it with the FP64 LU of its FP64 matrix
// (factored in place; the next solve assembles it again); then redoes its post-processing.  Runs
// synchronously on the plan's stream; requests that passed are not touched.
int rescue(tvlm_vlm_plan* P) {
    const int B = P->active;
    const int64_t N = P->N, NN = N * N;
    hipStream_t st = P->stream;
    std::vector<int32_t> conv(B), info(B);
    std::vector<double> berr(B);
    TVLM_HIP(hipMemcpyAsync(conv.data(), P->conv, sizeof(int32_t) * B, hipMemcpyDeviceToHost, st));
    TVLM_HIP(hipMemcpyAsync(info.data(), P->info, sizeof(int32_t) * B, hipMemcpyDeviceToHost, st));
    TVLM_HIP(hipMemcpyAsync(berr.data(), P->berr, sizeof(double) * B, hipMemcpyDeviceToHost, st));
    TVLM_HIP(hipStreamSynchronize(st));
    for (int b = 0; b < B; b++) {
        P->st_berr[b] = berr[b];
        if (conv[b]) continue;
        double* A64 = P->lhs + b * NN;
        float* A32 = P->lhs32 + b * NN;
        int32_t* ipiv = P->ipiv + b * N;
        int32_t* inf = P->info + b;
        double* x = P->x + b * N;
        double* rhs = P->rhs + b * N;
        double* res = P->res + b * N;
        float* r32 = P->r32 + b * N;
        tvlm_view L32 = {A32, {N, N, 1}, {1, N, NN}};
        tvlm_view R32 = {r32, {N, 1, 1}, {1, N, N}};
        const dim3 rg((unsigned)((N + kResidRows - 1) / kResidRows), 1);
        int32_t status = 0, corr = P->st_corr[b];
        if (info[b] == kGetrfStalled) {
            hipLaunchKernelGGL(k_to_f32, dim3(grid_for(NN)), dim3(256), 0, st, A64, A32, NN);
            TVLM_LAUNCHED();
            TVLM_TRY(getrf_single_group_f32(&L32, ipiv, inf, st));
            TVLM_TRY(tvlm_fill_f64(0, x, 1, 0.0, N, st));
            TVLM_HIP(hipMemcpyAsync(res, rhs, sizeof(double) * N, hipMemcpyDeviceToDevice, st));
            status |= kStRefactored;
            corr = 0;
        }
        bool ok = false;
        while (corr < kMaxCorrections && !ok) {
            hipLaunchKernelGGL(k_to_f32, dim3(grid_for(N)), dim3(256), 0, st, res, r32, N);
            TVLM_LAUNCHED();
            TVLM_TRY(tvlm_getrs_f32(&L32, ipiv, &R32, st));
            hipLaunchKernelGGL(k_add_f32, dim3(grid_for(N)), dim3(256), 0, st, x, r32, N);
            TVLM_LAUNCHED();
            corr++;
            hipLaunchKernelGGL(k_residual<false>, rg, dim3(kResidRows * kResidWaves), 0, st, A64, (int)N, rhs, x, res,
                               P->rowabs + b * N);
            TVLM_LAUNCHED();
            hipLaunchKernelGGL(k_refine_check, dim3(1), dim3(256), 0, st, res, x, P->rowabs + b * N, inf, (int)N,
                               P->berr + b, P->conv + b);
            TVLM_LAUNCHED();
            int32_t c = 0;
            TVLM_HIP(hipMemcpyAsync(&c, P->conv + b, sizeof(int32_t), hipMemcpyDeviceToHost, st));
            TVLM_HIP(hipMemcpyAsync(&P->st_berr[b], P->berr + b, sizeof(double), hipMemcpyDeviceToHost, st));
            TVLM_HIP(hipStreamSynchronize(st));
            ok = c != 0;
        }
        if (ok) {
            if (corr > kRefine + 1) status |= kStMoreCorrections;
        } else {
            // the plain path's solve of this request: FP64 LU of its FP64 matrix, in place
            tvlm_view L64 = {A64, {N, N, 1}, {1, N, NN}};
            TVLM_TRY(tvlm_getrf_f64(&L64, ipiv, inf, st));
            int32_t i64 = 0;
            TVLM_HIP(hipMemcpyAsync(&i64, inf, sizeof(int32_t), hipMemcpyDeviceToHost, st));
            TVLM_HIP(hipStreamSynchronize(st));
            if (i64 == kGetrfStalled) {
                // its factors are invalid and the matrix is gone: assemble it again, one-group panels
                TVLM_TRY(matrix(P, b, true));
                TVLM_TRY(getrf_single_group_f64(&L64, ipiv, inf, st));
                TVLM_HIP(hipMemcpyAsync(&i64, inf, sizeof(int32_t), hipMemcpyDeviceToHost, st));
                TVLM_HIP(hipStreamSynchronize(st));
                status |= kStRefactored;
            }
            TVLM_HIP(hipMemcpyAsync(x, rhs, sizeof(double) * N, hipMemcpyDeviceToDevice, st));
            tvlm_view X = {x, {N, 1, 1}, {1, N, N}};
            TVLM_TRY(tvlm_getrs_f64(&L64, ipiv, &X, st));
            status |= kStFallback64;
            if (i64 != 0) status |= kStUnresolved;
            P->st_berr[b] = NAN;  // the FP64 matrix is factored in place: no residual against it
        }
        P->st_status[b] = status;
        P->st_corr[b] = corr;
        TVLM_TRY(post(P, b, 1));
    }
    return TVLM_OK;
}

}  // namespace
}  // namespace tvlm

using namespace tvlm;

extern "C" {

int tvlm_vlm_create(tvlm_vlm_plan** plan, int32_t n_surf, const int64_t* ns, const int64_t* nc,
                    const double* const* verts_init, int32_t batch, int32_t mode, void* stream) {
    TVLM_REQUIRE(plan && ns && nc && verts_init, "null argument");
    TVLM_REQUIRE(n_surf >= 1 && n_surf <= kMaxS, "n_surf %d out of range", n_surf);
    TVLM_REQUIRE(batch >= 1 && batch <= 4096, "batch %d out of range", batch);
    TVLM_REQUIRE(mode == 0 || mode == 1, "mode must be 0 (plain FP64) or 1 (served)");
    auto* P = new tvlm_vlm_plan();
    P->mode = mode;
    P->n_surf = n_surf;
    P->batch = batch;
    P->stream = as_stream(stream);
    int64_t N = 0;
    for (int m = 0; m < n_surf; m++) {
        if (ns[m] < 1 || nc[m] < 1) {
            delete P;
            set_error("surface %d: empty mesh", m);
            return TVLM_ERR_INVALID;
        }
        P->ns[m] = ns[m];
        P->nc[m] = nc[m];
        P->off[m] = N;
        P->vsz[m] = (ns[m] + 1) * (nc[m] + 1) * 4;
        P->wsz[m] = (ns[m] + 1) * 2 * 4;
        P->psz[m] = ns[m] * nc[m];
        N += ns[m] * nc[m];
    }
    P->N = (int32_t)N;
    const int64_t NN = N * N;
    const int64_t nb = mode == 1 ? batch : 1;  // plain mode reuses one matrix for every request
    auto fail = [&](int rc) {
        (void)tvlm_lhs_group_destroy(P->group);
        for (void* p : P->allocs) (void)hipFree(p);
        if (P->par_host) (void)hipHostFree(P->par_host);
        if (P->done) (void)hipEventDestroy(P->done);
        delete P;
        return rc;
    };
    int rc = TVLM_OK;
    for (int m = 0; m < n_surf && rc == TVLM_OK; m++) {
        const size_t v = sizeof(double) * P->vsz[m], p3 = sizeof(double) * 3 * P->psz[m], p1 = sizeof(double) * P->psz[m];
        rc = P->alloc((void**)&P->init[m], v);
        if (rc == TVLM_OK) rc = P->alloc((void**)&P->verts[m], v * batch);
        if (rc == TVLM_OK) rc = P->alloc((void**)&P->wake[m], sizeof(double) * P->wsz[m] * batch);
        if (rc == TVLM_OK) rc = P->alloc((void**)&P->colloc[m], p3 * batch);
        if (rc == TVLM_OK) rc = P->alloc((void**)&P->normals[m], p3 * batch);
        if (rc == TVLM_OK) rc = P->alloc((void**)&P->areas[m], p1 * batch);
        if (rc == TVLM_OK) rc = P->alloc((void**)&P->vel[m], p3 * batch);
        if (rc == TVLM_OK) rc = P->alloc((void**)&P->forces[m], p3 * batch);
        if (rc == TVLM_OK) rc = P->alloc((void**)&P->gdelta[m], p1 * batch);
        if (rc == TVLM_OK) rc = tvlm_copy(0, P->init[m], 1, 1, verts_init[m], 1, sizeof(double), P->vsz[m], stream);
    }
    if (rc == TVLM_OK) rc = P->alloc((void**)&P->lhs, sizeof(double) * NN * nb);
    if (rc == TVLM_OK && mode == 1) {  // prep stands behind lhs32 (an allocation of its own takes 0.1 ms)
        const size_t prep = getrs_prep_bytes_f32(N, batch), at = (sizeof(float) * NN * nb + 255) / 256 * 256;
        rc = P->alloc((void**)&P->lhs32, at + prep);
        if (rc == TVLM_OK && prep) P->prep = reinterpret_cast<char*>(P->lhs32) + at;
    }
    if (rc == TVLM_OK && mode == 1) rc = P->alloc((void**)&P->r32, sizeof(float) * N * batch);
    if (rc == TVLM_OK && mode == 1) rc = P->alloc((void**)&P->res, sizeof(double) * N * batch);
    if (rc == TVLM_OK && mode == 1) rc = P->alloc((void**)&P->rowabs, sizeof(double) * N * batch);
    if (rc == TVLM_OK && mode == 1) rc = P->alloc((void**)&P->berr, sizeof(double) * batch);
    if (rc == TVLM_OK && mode == 1) rc = P->alloc((void**)&P->conv, sizeof(int32_t) * batch);
    if (rc == TVLM_OK) rc = P->alloc((void**)&P->rhs, sizeof(double) * N * batch);
    if (rc == TVLM_OK) rc = P->alloc((void**)&P->x, sizeof(double) * N * batch);
    if (rc == TVLM_OK) rc = P->alloc((void**)&P->par, sizeof(double) * (16 * n_surf + kPar) * batch);
    if (rc == TVLM_OK) rc = P->alloc((void**)&P->coef, sizeof(double) * 8 * n_surf * batch);
    if (rc == TVLM_OK) rc = P->alloc((void**)&P->ipiv, sizeof(int32_t) * N * nb);
    if (rc == TVLM_OK) rc = P->alloc((void**)&P->info, sizeof(int32_t) * batch);
    if (rc == TVLM_OK) {
        hipError_t e = hipHostMalloc((void**)&P->par_host, sizeof(double) * (16 * n_surf + kPar) * batch,
                                     hipHostMallocDefault);
        if (e != hipSuccess) {
            set_error("hipHostMalloc failed: %s", hipGetErrorString(e));
            rc = TVLM_ERR_NOMEM;
        }
    }
    if (rc == TVLM_OK && hipEventCreateWithFlags(&P->done, hipEventDisableTiming) != hipSuccess) {
        set_error("hipEventCreateWithFlags failed");
        rc = TVLM_ERR_HIP;
    }
    if (rc == TVLM_OK && hipEventRecord(P->done, P->stream) != hipSuccess) {
        set_error("hipEventRecord failed");
        rc = TVLM_ERR_HIP;
    }
    if (rc == TVLM_OK && mode == 1) {
        // the grouped assembly's work list: request b's matrix and surfaces (iteration 1: one wake row)
        std::vector<tvlm_lhs_item> items(batch);
        std::vector<tvlm_view> vv((size_t)batch * n_surf * 8);
        for (int b = 0; b < batch; b++) {
            tvlm_view *V = &vv[((size_t)b * 8 + 0) * n_surf], *W = &vv[((size_t)b * 8 + 1) * n_surf],
                      *C = &vv[((size_t)b * 8 + 2) * n_surf], *Nn = &vv[((size_t)b * 8 + 3) * n_surf];
            for (int m = 0; m < n_surf; m++) {
                tvlm_view A, VEL, F, GD;
                views(P, b, m, V[m], W[m], C[m], Nn[m], A, VEL, F, GD);
            }
            items[b] = {{P->lhs + b * NN, {N, N, 1}, {1, N, NN}}, n_surf, C, Nn, V, W, 1};
        }
        rc = tvlm_lhs_group_create(&P->group, batch, items.data(), stream);
    }
    if (rc != TVLM_OK) return fail(rc);
    *plan = P;
    return TVLM_OK;
}

int tvlm_vlm_solve(tvlm_vlm_plan* P, const double* alpha, const double* beta, double u_inf, double rho,
                   const double* cm_ref) {
    TVLM_REQUIRE(P, "null plan");
    return tvlm_vlm_solve_n(P, P->batch, alpha, beta, u_inf, rho, cm_ref);
}

int tvlm_vlm_solve_n(tvlm_vlm_plan* P, int32_t n_active, const double* alpha, const double* beta, double u_inf,
                     double rho, const double* cm_ref) {
    TVLM_REQUIRE(P && alpha, "null argument");
    TVLM_REQUIRE(n_active >= 1 && n_active <= P->batch, "n_active %d out of range 1..%d", n_active, P->batch);
    const int n = P->n_surf, B = n_active;
    P->active = B;
    const double c0[3] = {cm_ref ? cm_ref[0] : 0.25, cm_ref ? cm_ref[1] : 0.0, cm_ref ? cm_ref[2] : 0.0};
    TVLM_HIP(hipEventSynchronize(P->done));  // the pinned parameters may still be read
    for (int b = 0; b < B; b++) {
        const double a = alpha[b], be = beta ? beta[b] : 0.0, u = u_inf;
        double* T = P->par_host + (int64_t)b * (16 * n + kPar);
        // translation by -100 u (cos a, 0, sin a): 100-chord wake row (vlm.cpp:104-108)
        const double tx = -100.0 * u * std::cos(a), tz = -100.0 * u * std::sin(a);
        for (int m = 0; m < n; m++, T += 16) {
            for (int k = 0; k < 16; k++) T[k] = (k % 5 == 0) ? 1.0 : 0.0;
            T[12] = tx;
            T[14] = tz;
        }
        const double fs[3] = {u * std::cos(a) * std::cos(be), -u * std::cos(a) * std::sin(be), u * std::sin(a)};
        // lift axis normalize(fs x y) (vlm/src/vlm_utils.cpp:13-15)
        const double ln = std::sqrt(fs[2] * fs[2] + fs[0] * fs[0]);
        const double v[kPar] = {a,          fs[0], fs[1],      fs[2],           -fs[2] / ln, 0.0,
                                fs[0] / ln, c0[0] + tx, c0[1], c0[2] + tz,
                                0.5 * rho * (fs[0] * fs[0] + fs[1] * fs[1] + fs[2] * fs[2]), 0.0};
        std::copy(v, v + kPar, T);
    }
    hipStream_t st = P->stream;
    TVLM_HIP(hipMemcpyAsync(P->par, P->par_host, sizeof(double) * (16 * n + kPar) * B, hipMemcpyHostToDevice, st));
    TVLM_TRY(geometry(P, 0, B));
    const int64_t N = P->N, NN = N * N;
    if (P->mode == 0) {
        tvlm_view L = {P->lhs, {N, N, 1}, {1, N, NN}};
        for (int b = 0; b < B; b++) {
            TVLM_TRY(matrix(P, b, false));
            TVLM_TRY(tvlm_getrf_f64(&L, P->ipiv, P->info + b, st));
            TVLM_HIP(hipMemcpyAsync(P->x + b * N, P->rhs + b * N, sizeof(double) * N, hipMemcpyDeviceToDevice, st));
            tvlm_view X = {P->x + b * N, {N, 1, 1}, {1, N, N}};
            TVLM_TRY(tvlm_getrs_f64(&L, P->ipiv, &X, st));
        }
        TVLM_TRY(post(P, 0, B));
    } else {
        // every request's matrix and its FP32 copy in one grouped launch
        TVLM_TRY(lhs_group_assign_seeded(P->group, B, P->lhs, P->lhs32, st));
        tvlm_view L32 = {P->lhs32, {N, N, B}, {1, N, NN}};
        TVLM_TRY(tvlm_getrf_f32(&L32, P->ipiv, P->info, st));
        TVLM_TRY(getrs_prepare_f32(&L32, P->ipiv, P->prep, st));
        tvlm_view R32 = {P->r32, {N, 1, B}, {1, N, N}};
        // x = 0, r = b; then kRefine + 1 corrections x += A32^{-1} r, r = b - A64 x
        TVLM_TRY(tvlm_fill_f64(0, P->x, 1, 0.0, N * B, st));
        const dim3 rg((unsigned)((N + kResidRows - 1) / kResidRows), B);
        for (int it = 0; it <= kRefine; it++) {
            if (it == 0) {
                hipLaunchKernelGGL(k_to_f32, dim3(grid_for(N * B)), dim3(256), 0, st, P->rhs, P->r32, N * B);
            } else {
                if (it == 1)
                    hipLaunchKernelGGL(k_residual<true>, rg, dim3(kResidRows * kResidWaves), 0, st, P->lhs, (int)N,
                                       P->rhs, P->x, P->res, P->rowabs);
                else
                    hipLaunchKernelGGL(k_residual<false>, rg, dim3(kResidRows * kResidWaves), 0, st, P->lhs, (int)N,
                                       P->rhs, P->x, P->res, P->rowabs);
                TVLM_LAUNCHED();
                hipLaunchKernelGGL(k_to_f32, dim3(grid_for(N * B)), dim3(256), 0, st, P->res, P->r32, N * B);
            }
            TVLM_LAUNCHED();
            TVLM_TRY(getrs_prepared_f32(&L32, P->ipiv, P->prep, &R32, st));
            hipLaunchKernelGGL(k_add_f32, dim3(grid_for(N * B)), dim3(256), 0, st, P->x, P->r32, N * B);
            TVLM_LAUNCHED();
        }
        // the returned x of every request: its residual and the convergence test (the rescue of the
        // requests that fail it runs in tvlm_vlm_results)
        hipLaunchKernelGGL(k_residual<false>, rg, dim3(kResidRows * kResidWaves), 0, st, P->lhs, (int)N, P->rhs, P->x,
                           P->res, P->rowabs);
        TVLM_LAUNCHED();
        hipLaunchKernelGGL(k_refine_check, dim3(B), dim3(256), 0, st, P->res, P->x, P->rowabs, P->info, (int)N,
                           P->berr, P->conv);
        TVLM_LAUNCHED();
        TVLM_TRY(post(P, 0, B));
    }
    TVLM_HIP(hipEventRecord(P->done, st));
    P->solved = true;
    P->checked = false;
    P->st_status.assign(B, 0);
    P->st_corr.assign(B, P->mode == 1 ? kRefine + 1 : 0);
    P->st_berr.assign(B, 0.0);
    return TVLM_OK;
}

// Waits for the plan's last solve.  cl[n], cm[n][3], gamma[n][N], info[n] for the n requests of
// the last solve; null pointers are skipped.  The copies are queued on the plan's stream (not the
// null stream), so reading one plan's results does not wait for work on other streams.
int tvlm_vlm_results(tvlm_vlm_plan* P, double* cl, double* cm, double* gamma, int32_t* info) {
    TVLM_REQUIRE(P && P->solved, "no solve has run on this plan");
    const int n = P->n_surf, B = P->active;
    hipStream_t st = P->stream;
    if (P->mode == 1 && !P->checked) {
        TVLM_TRY(rescue(P));
        P->checked = true;
    }
    std::vector<double> coef((size_t)8 * n * B);
    TVLM_HIP(hipMemcpyAsync(coef.data(), P->coef, sizeof(double) * coef.size(), hipMemcpyDeviceToHost, st));
    if (gamma) TVLM_HIP(hipMemcpyAsync(gamma, P->x, sizeof(double) * P->N * B, hipMemcpyDeviceToHost, st));
    if (info) TVLM_HIP(hipMemcpyAsync(info, P->info, sizeof(int32_t) * B, hipMemcpyDeviceToHost, st));
    TVLM_HIP(hipEventRecord(P->done, st));
    TVLM_HIP(hipEventSynchronize(P->done));
    for (int b = 0; b < B; b++) {
        // per surface: cf[2] = sum(F . l) / q and cf[3..5] = sum(r x F) / q (q = rho |V|^2 / 2,
        // vlm_backend_cpu.cpp:323-362); CL area-weighted, CM area*MAC-weighted over the surfaces
        double cl_sum = 0.0, area_sum = 0.0, mac_sum = 0.0, cm_sum[3] = {0.0, 0.0, 0.0};
        for (int m = 0; m < n; m++) {
            const double* cf = coef.data() + ((size_t)b * n + m) * 8;
            cl_sum += cf[2];
            for (int k = 0; k < 3; k++) cm_sum[k] += cf[3 + k];
            area_sum += cf[0];
            mac_sum += cf[1];
        }
        if (cl) cl[b] = cl_sum / area_sum;
        if (cm)
            for (int k = 0; k < 3; k++) cm[3 * b + k] = cm_sum[k] / (area_sum * mac_sum);
    }
    return TVLM_OK;
}

// What the served refinement took for each request of the last solve (after tvlm_vlm_results).
int tvlm_vlm_refinement(tvlm_vlm_plan* P, int32_t* status, int32_t* corrections, double* backward_error) {
    TVLM_REQUIRE(P && P->solved, "no solve has run on this plan");
    if (P->mode == 1 && !P->checked) {
        TVLM_TRY(rescue(P));
        P->checked = true;
    }
    const int B = P->active;
    for (int b = 0; b < B; b++) {
        if (status) status[b] = P->st_status[b];
        if (corrections) corrections[b] = P->st_corr[b];
        if (backward_error) backward_error[b] = P->st_berr[b];
    }
    return TVLM_OK;
}

// Moves the plan to another stream: later solves queue on `stream`, after the plan's own latest
// work on its previous stream (a device-side wait on the plan's event; the host does not block, and
// whatever else runs on the previous stream is not waited for).
int tvlm_vlm_set_stream(tvlm_vlm_plan* P, void* stream) {
    TVLM_REQUIRE(P, "null plan");
    if (as_stream(stream) == P->stream) return TVLM_OK;
    TVLM_HIP(hipStreamWaitEvent(as_stream(stream), P->done, 0));
    P->stream = as_stream(stream);
    return TVLM_OK;
}

// *done = 1 once the plan's latest work has finished (does not block)
int tvlm_vlm_query(const tvlm_vlm_plan* P, int32_t* done) {
    TVLM_REQUIRE(P && done, "null argument");
    const hipError_t e = hipEventQuery(P->done);
    *done = e == hipSuccess ? 1 : 0;
    if (e != hipErrorNotReady) TVLM_HIP(e);
    return TVLM_OK;
}

int tvlm_vlm_footprint(const tvlm_vlm_plan* P, int64_t* device_bytes) {
    TVLM_REQUIRE(P && device_bytes, "null argument");
    *device_bytes = P->bytes;
    return TVLM_OK;
}

int tvlm_vlm_destroy(tvlm_vlm_plan* P) {
    if (!P) return TVLM_OK;
    (void)hipEventSynchronize(P->done);
    (void)tvlm_lhs_group_destroy(P->group);
    for (void* p : P->allocs) (void)hipFree(p);
    (void)hipEventDestroy(P->done);
    if (P->par_host) (void)hipHostFree(P->par_host);
    delete P;
    return TVLM_OK;
}

}  // extern "C"
