// tvlm_lu.hip -- dense LU with partial pivoting (getrf) and solve (getrs) on gfx950.
//
// Semantics follow LAPACK ?getrf/?getrs as called by the reference (vlm_backend_cpu_lapack.cpp:40-94):
// column-major in place L\U, unit lower L, 1-based ipiv, pivot = first row of max |a| in the
// column, info = first exactly-zero pivot (1-based), factorisation continues past it.
//
// getrf is blocked right-looking; each panel (64 columns, 32 while more than 2048 rows remain):
//   1. k_panel_spec : the panel with the pivots of a few candidate rows, checked against all rows (three
//                     rounds); the matrices for which no round stood take
//      k_panel_reg  : one work-group factors the panel (register-resident sub-panels, DPP argmax,
//                     LDS-only barriers) and lists the panel's composed row interchanges; panels
//                     of more than 1024 rows of one matrix (or of a few) are factored by several
//                     work-groups together instead (k_panel_coop, 64 columns, one exchange through
//                     global memory per column);
//   2. k_swap_trsm  : the interchanges on the columns left and right of the panel, and
//                     U12 = L11^{-1} A12 for the columns right of it, on the matrix cores;
//   3. k_update     : A22 -= L21 U12 on the matrix cores (double-buffered 16-deep k-slices).
// Panels taller than the cooperative groups hold (and taller than 8192 rows) use the
// column-by-column k_panel + k_laswp + k_trsm instead.
// getrs (n <= 16384): the interchanges are composed (k_solve_prep per block of 64 pivots, k_solve_compose
// over the blocks) and the 64 x 64 diagonal blocks of L and U inverted (k_solve_prep); then up to n = 256 one
// work-group per right-hand side does the rest (k_solve_small).  Above that solve_route chooses: a work-group per
// right-hand side in 64-row steps (k_solve_blocked), or the interchanges first (k_solve_perm) and each step of
// a substitution on all trailing row blocks at once (k_trsv_step by 256 rows, k_trsv_block by 64), or, with
// many right-hand sides, 64-row steps that multiply all of them on the matrix cores (k_inv_apply, k_update); larger
// n uses block-row kernels (k_diag_solve / k_off_update).
#include <atomic>
#include <map>
#include <utility>
#include <mutex>
#include <type_traits>
#include <vector>

#include <hip/hip_ext.h>

#include "tvlm_internal.hpp"

namespace tvlm {
namespace {

constexpr int kPanelThreads = 1024;
constexpr int NB = 64;


template <typename T>
__global__ __launch_bounds__(kPanelThreads) void k_panel(T* __restrict__ a, int64_t lda, int n, int k0, int kb,
                                                         int32_t* __restrict__ ipiv, int32_t* __restrict__ info) {
    __shared__ T sval[kPanelThreads];
    __shared__ int sidx[kPanelThreads];
    __shared__ T srow[NB];
    const int t = threadIdx.x;
    for (int k = k0; k < k0 + kb; k++) {
        T* colk = a + (int64_t)k * lda;
        // pivot search: max |a(i,k)|, i >= k, first index on ties
        T best = T(-1);
        int bi = k;
        for (int i = k + t; i < n; i += kPanelThreads) {
            const T v = fabs(colk[i]);
            if (v > best) {
                best = v;
                bi = i;
            }
        }
        sval[t] = best;
        sidx[t] = bi;
        __syncthreads();
        for (int s = kPanelThreads / 2; s > 0; s >>= 1) {
            if (t < s) {
                const T v2 = sval[t + s];
                const int i2 = sidx[t + s];
                if (v2 > sval[t] || (v2 == sval[t] && i2 < sidx[t])) {
                    sval[t] = v2;
                    sidx[t] = i2;
                }
            }
            __syncthreads();
        }
        const int p = sidx[0];
        if (t == 0) ipiv[k] = p + 1;
        // swap rows k and p inside the panel columns, and stage the pivot row
        if (t < kb) {
            const int j = k0 + t;
            T* cj = a + (int64_t)j * lda;
            const T vk = cj[k], vp = cj[p];
            if (p != k) {
                cj[k] = vp;
                cj[p] = vk;
            }
            srow[t] = (p != k) ? vp : vk;
        }
        __syncthreads();
        const T piv = srow[k - k0];
        if (t == 0 && piv == T(0) && info[0] == 0) info[0] = k + 1;
        if (piv != T(0)) {
            const T r = T(1) / piv;
            for (int i = k + 1 + t; i < n; i += kPanelThreads) {
                const T l = colk[i] * r;
                colk[i] = l;
                for (int j = k + 1; j < k0 + kb; j++) {
                    T* cj = a + (int64_t)j * lda;
                    cj[i] -= l * srow[j - k0];
                }
            }
        }
        __syncthreads();
    }
}

// Apply interchanges ipiv[k0 .. k0+kb) to columns [c0, c1) (one thread per column).
template <typename T>
__global__ void k_laswp(T* __restrict__ a, int64_t lda, int c0, int c1, int k0, int kb, const int32_t* __restrict__ ipiv) {
    const int j = c0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= c1) return;
    T* cj = a + (int64_t)j * lda;
    for (int k = k0; k < k0 + kb; k++) {
        const int p = ipiv[k] - 1;
        if (p != k) {
            const T t = cj[k];
            cj[k] = cj[p];
            cj[p] = t;
        }
    }
}

// U12 = L11^{-1} A12 for columns [j0, n), L11 = unit lower of a(k0:k0+kb, k0:k0+kb).
template <typename T>
__global__ __launch_bounds__(256) void k_trsm(T* __restrict__ a, int64_t lda, int n, int k0, int kb, int j0) {
    __shared__ T L[NB][NB + 1];
    for (int e = threadIdx.x; e < kb * kb; e += blockDim.x) {
        const int r = e % kb, c = e / kb;
        L[r][c] = a[(k0 + r) + (int64_t)(k0 + c) * lda];
    }
    __syncthreads();
    const int j = j0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    T* cj = a + (int64_t)j * lda + k0;
    T x[NB];
#pragma unroll
    for (int r = 0; r < NB; r++)
        if (r < kb) x[r] = cj[r];
#pragma unroll
    for (int c = 0; c < NB; c++) {
        if (c < kb) {
            const T xc = x[c];
#pragma unroll
            for (int r = c + 1; r < NB; r++)
                if (r < kb) x[r] -= L[r][c] * xc;
        }
    }
#pragma unroll
    for (int r = 0; r < NB; r++)
        if (r < kb) cj[r] = x[r];
}

// ---- fast getrf: register-resident panel, fused interchange + TRSM, MFMA trailing update ------
//
// k_panel_reg: one work-group of NT threads factors the panel rows [k0, n) x columns [k0, k0+kb),
// kb <= NB.  Thread t owns rows k0 + t + NT q (q < Q).  The panel is processed left-looking in
// sub-panels of IB columns held in registers (Q x IB values per thread): a sub-panel first receives
// the updates of the panel's earlier sub-panels (blocked forward substitution with the inverses of
// their unit-lower IB x IB diagonal blocks, kept in LDS), then is factored column by column with
// partial pivoting (argmax by wave shuffles + one LDS exchange, first index on ties; the pivot row
// and row k exchange through LDS; reciprocal scaling and rank-1 update in registers).  Inside the
// column loop only LDS is touched and the work-group synchronises with an LDS-only barrier, so no
// step waits for global memory; pivots stay in LDS until the panel ends.  Each sub-panel's
// interchanges reach the panel's other columns as one gather / scatter, and at the end thread 0
// composes the panel's interchanges into (destination, source) row pairs for the rest of the matrix.

constexpr int kPermInts = 1 + 2 * 2 * NB;  // composed interchanges of one panel

// barrier for LDS traffic only: waits for this wave's LDS operations, not for global memory
__device__ __forceinline__ void lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <typename T>
__device__ __forceinline__ void argmax_merge(T& best, int& bi, T v, int i) {
    const bool take = (v > best) | ((v == best) & (i < bi));
    best = take ? v : best;
    bi = take ? i : bi;
}

// One DPP step of a wave argmax: the value and index of the lane CTRL selects (row_shr / row_bcast
// within the row and bank masks) are merged in; lanes without a source keep their own pair.
template <int CTRL, int ROWM>
__device__ __forceinline__ void dpp_argmax_step(double& v, int& i) {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const int olo = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWM, 0xf, false);
    const int ohi = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWM, 0xf, false);
    const int oi = __builtin_amdgcn_update_dpp(i, i, CTRL, ROWM, 0xf, false);
    argmax_merge(v, i, __hiloint2double(ohi, olo), oi);
}
template <int CTRL, int ROWM>
__device__ __forceinline__ void dpp_argmax_step(float& v, int& i) {
    const int ov = __builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL, ROWM, 0xf, false);
    const int oi = __builtin_amdgcn_update_dpp(i, i, CTRL, ROWM, 0xf, false);
    argmax_merge(v, i, __int_as_float(ov), oi);
}
__device__ __forceinline__ double readlane63(double v) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), 63),
                            __builtin_amdgcn_readlane(__double2loint(v), 63));
}
__device__ __forceinline__ float readlane63(float v) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
// wave-wide argmax (larger value, then smaller index), result in every lane: row_shr 1, 2, 4, 8
// gathers each row's maximum into its lane 15, row_bcast 15 / 31 carry it across rows to lane 63
template <typename T>
__device__ __forceinline__ void wave_argmax(T& v, int& i) {
    dpp_argmax_step<0x111, 0xf>(v, i);
    dpp_argmax_step<0x112, 0xf>(v, i);
    dpp_argmax_step<0x114, 0xf>(v, i);
    dpp_argmax_step<0x118, 0xf>(v, i);
    dpp_argmax_step<0x142, 0xa>(v, i);
    dpp_argmax_step<0x143, 0xc>(v, i);
    v = readlane63(v);
    i = __builtin_amdgcn_readlane(i, 63);
}

// Composes the interchanges pos[i] <-> piv[i] (i < cnt <= 64, applied in order, piv[i] >= pos[i],
// positions [first, first + cnt)) into (dst, src) row pairs, using one wave: lane l holds the source
// row of position first + l, and the rows outside the block that the interchanges touch are kept as
// (position, source) entries, one per lane.  Every lane calls it; returns the pair count (<= 2 cnt).
__device__ int wave_compose_swaps(int first, int cnt, const int* piv, int* pd, int* ps) {
    const int lane = threadIdx.x & 63;
    int src = first + lane;  // position first + lane
    int okey = -1, oval = -1;
    int nout = 0;
    for (int i = 0; i < cnt; i++) {
        const int p = __builtin_amdgcn_readfirstlane(piv[i]);
        if (p == first + i) continue;
        const int vi = __builtin_amdgcn_readlane(src, i);
        if (p < first + cnt) {
            const int j = p - first;
            const int vj = __builtin_amdgcn_readlane(src, j);
            src = lane == i ? vj : (lane == j ? vi : src);
        } else {
            const unsigned long long m = __ballot(okey == p);
            int e;
            if (m != 0ull) {
                e = __ffsll((long long)m) - 1;
            } else {
                e = nout++;
                okey = lane == e ? p : okey;
                oval = lane == e ? p : oval;
            }
            const int ve = __builtin_amdgcn_readlane(oval, e);
            src = lane == i ? ve : src;
            oval = lane == e ? vi : oval;
        }
    }
    const bool in_pair = lane < cnt && src != first + lane;
    const bool out_pair = lane < nout && oval != okey;
    const unsigned long long mi = __ballot(in_pair), mo = __ballot(out_pair);
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const int ni = __popcll(mi);
    if (in_pair) {
        const int k = __popcll(mi & below);
        pd[k] = first + lane;
        ps[k] = src;
    }
    if (out_pair) {
        const int k = ni + __popcll(mo & below);
        pd[k] = okey;
        ps[k] = oval;
    }
    return ni + __popcll(mo);
}

// ---- speculative panel ----------------------------------------------------------------------------
// Partial pivoting has one exchange over all rows per column; on the influence matrices of wings
// nearly every pivot lies in the panel's diagonal block.  k_panel_spec factors a small set of
// candidate rows on its own, eliminates all other rows against the resulting U11 and checks that
// none of them would have been a pivot: every multiplier |l| < 1.  When that holds everywhere, the
// candidates' pivots are the ones partial pivoting over all rows picks, so nothing had to be exchanged.
// Three rounds:
//   round 1 (R = 1): candidates = the panel's kb diagonal rows, no interchange among them;
//   rounds 2, 3 (R = 2): only for matrices whose earlier rounds failed: plus up to 64 rows that broke
//                    the check in them, column by column the worst first (keys); not tried where round 1
//                    was broken in more than half of the columns.  A panel with at most 64 other rows has all of
//                    them as candidates of round 2, and no round 3.
// A column whose pivot is zero or not finite, a tie among candidates, an |l| above 1 or within its own rounding
// of 1 (a row larger than the pivot by an ulp can have |l| = 1; a tie is not settled by the row order) or a
// NaN fails the round.  Wings keep clear of that line (largest |l| 0.9992 over elliptic, swept and rectangular
// ones of 256 to 4096 panels).
// The rounds write their result to sp.w and leave the matrix as it is: the next round copies the
// result of one that stood, the panel kernel launched after them (k_panel_coop / k_panel_reg) copies
// round 3's, or factors the panel itself where all failed.  A matrix whose panels failed kSpecFails
// times in a row skips the rounds from then on, up to the panels whose rows are all candidates.
// On the influence matrices of rectangular and 25-degree swept wings every panel stands in round 1;
// on the elliptic ones (pivots at the tip panels, up to 1538 rows below the diagonal) all (16 x 16, 12 spans
// x 100), 7 of 17 (100 spans x 12), 3 of 30 (45 x 45) or none (64 x 64) do, most others in round 2 and, at 64 x
// 64, a quarter in round 3.
//
// Every work-group factors the candidates for itself (a 64-step chain in registers and LDS: one
// launch and no exchange) and then takes its share of the other rows, 16 per wave and step on the
// matrix cores: with Y = L21^T, 16 columns of the panel at a time, R_b = A_b^T - sum_{c<b} U_cb^T Y_c and
// Y_b = Uinv_bb^T R_b (Uinv_bb: inverse of the 16 x 16 diagonal block), then corrected once, Y_b += Uinv_bb^T
// (R_b - U_bb^T Y_b).  Without the correction the error of Y_b grows with the condition of U_bb (1e8: 1e-11 of the
// matrix in FP64), while its multipliers stay below 1; with it the factors are as accurate as column by column
// up to spec_condition_limit, past which the round fails.  The MFMA output layout is the
// second operand's layout, so the blocks chain without moving between lanes.  What bounds it is the
// candidates' chain, 64 dependent pivot steps.  Per 4096-row FP64 panel of one matrix, round 1 took 21 us
// (loads 2.3, chain 12.8, inverses and staging 2.8, rows 2.9; FP32 17 us) before the correction and a later
// round 52 us (its chain 41: the pivot search and v_readlane broadcasts); over all panels of such a matrix round 1
// takes 22.0 us without the correction and the condition, 23.6 with them.  The cooperative panel with an exchange
// per panel took 153 us, with an exchange per column 327 us.
typedef float vf4 __attribute__((ext_vector_type(4)));
typedef double vd4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Mf16;
template <>
struct Mf16<float> {
    typedef vf4 vacc;
    static __device__ __forceinline__ vacc mfma(float p, float q, vacc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(p, q, c, 0, 0, 0);
    }
    // row of D in register r of lane l; also the k index lane l stands for when register r of a
    // result is the second operand (the contraction may run in any order, the same in both operands)
    static __device__ __forceinline__ int k(int l, int r) { return 4 * (l >> 4) + r; }
};
template <>
struct Mf16<double> {
    typedef vd4 vacc;
    static __device__ __forceinline__ vacc mfma(double p, double q, vacc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(p, q, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int k(int l, int r) { return (l >> 4) + 4 * r; }
};

constexpr int kSpecFails = 2;  // failed panels in a row after which a matrix skips the rounds
// Rows that round 1 keeps per column: the one breaking the check by most among the row tiles of 16
// with index i mod kSpecSlots.  A wing's tip rows break it in a handful of columns (up to 6), in each of
// which the next pivots are mostly among its top rows: with one row per column 39 of the 63 panels of the
// elliptic 64 x 64 wing need round 3, with these 17.
constexpr int kSpecSlots = 16;
constexpr int kSpecRounds = 3;
// Columns with such a row past which rounds 2 and 3 are not tried: their candidates cannot hold all the pivots (a
// wing breaks at most 8, a matrix without a dominant diagonal nearly all; two failed rounds of 256 rows and
// more took 100 us).
constexpr int kSpecMaxBroken = NB / 2;
// Panels of at most this many rows have no rounds: k_panel_reg takes 1.6 us a column, a round's chain the same
// whatever the width.  With more matrices than CUs k_panel_reg, of which a CU holds several, gains: 1000 FP32
// matrices without a dominant diagonal, 40 x 40: 93 us without rounds, 130 with; 64 x 64 in FP64: 312 and 247.
template <typename T>
constexpr int spec_min_rows(int64_t batch) {
    return batch <= 256 ? 32 : sizeof(T) == 8 ? 48 : 64;
}
constexpr int kSpecMaxRows = 32768;  // rows of a panel (the cooperative panels hold no more)

// Buffers of one panel's speculative rounds (device); sets are zeroed once per factorisation.
template <typename T>
struct SpecBufs {
    bool on = false;
    T* w = nullptr;                      // results: matrix z at w + z ldw NB, {rows, NB} column-major
    int64_t ldw = 0;
    // this panel's [kSpecRounds - 1][batch][kSpecSlots][NB]: largest |l| > 1, with its row (null for a panel
    // whose other rows are all candidates of round 2)
    unsigned long long* keys = nullptr;
    int rounds = kSpecRounds;   // rounds of this panel
    int32_t* fail = nullptr;    // this panel's [kSpecRounds][batch]: 1 where the round failed, 2 in round 1
                                // where its blocks' condition failed it (then no row was checked)
    int32_t* ostate = nullptr;  // [batch]: failed panels in a row
    int batch = 1;
};

// The round (1-based) whose result stands for matrix z among the first `rounds`, 0 if none.
template <typename T>
__device__ __forceinline__ int spec_stood(const SpecBufs<T>& sp, int z, int rounds) {
    for (int r = 0; r < rounds; r++)
        if (sp.fail[r * sp.batch + z] == 0) return r + 1;
    return 0;
}

// Whether one of the rounds stood for matrix z (the failure count is kept by the one `keeper` thread).
template <typename T>
__device__ __forceinline__ bool spec_settled(const SpecBufs<T>& sp, int z, bool keeper) {
    const bool ok = spec_stood(sp, z, sp.rounds) != 0;
    if (keeper) {
        if (ok)
            sp.ostate[z] = 0;
        else if (sp.ostate[z] < kSpecFails)
            sp.ostate[z]++;
    }
    return ok;
}

// Copies a round's result into the panel; thread id of count (whole waves, 64 rows x 8 columns each at a time).
template <typename T>
__device__ __forceinline__ void spec_commit(const SpecBufs<T>& sp, int z, T* a, int64_t lda, int n, int k0, int kb,
                                            int id, int count) {
    const T* w = sp.w + (int64_t)z * sp.ldw * NB;
    const int m = n - k0;
    for (int e = id >> 6; e < (m + 63) / 64 * (NB / 8); e += count >> 6) {
        const int r = e / (NB / 8) * 64 + (id & 63), j0 = e % (NB / 8) * 8;
        T v[8];
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (r < m && j0 + j < kb) v[j] = w[r + (int64_t)(j0 + j) * sp.ldw];
#pragma unroll
        for (int j = 0; j < 8; j++)
            if (r < m && j0 + j < kb) a[(k0 + r) + (int64_t)(k0 + j0 + j) * lda] = v[j];
    }
}

__device__ __forceinline__ double lane_value(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
__device__ __forceinline__ float lane_value(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// 1/v to about an ulp (the hardware estimate and Newton steps); spec_pivot_ok bounds v so that none of
// the steps overflows.
__device__ __forceinline__ double spec_recip(double v) {
    double y = __builtin_amdgcn_rcp(v);
    y = fma(y, fma(-v, y, 1.0), y);
    return fma(y, fma(-v, y, 1.0), y);
}
__device__ __forceinline__ float spec_recip(float v) {
    const float y = __builtin_amdgcn_rcpf(v);
    return fmaf(y, fmaf(-v, y, 1.0f), y);
}
__device__ __forceinline__ bool spec_pivot_ok(double v) { return fabs(v) > 1e-290 && fabs(v) < 1e290; }
__device__ __forceinline__ bool spec_pivot_ok(float v) { return fabsf(v) > 1e-30f && fabsf(v) < 1e30f; }

// Lane N of every row of 16 lanes, to the whole row.
template <int N>
__device__ __forceinline__ double row_value(double v) {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    return __hiloint2double(__builtin_amdgcn_update_dpp(hi, hi, 0x150 + N, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(lo, lo, 0x150 + N, 0xf, 0xf, true));
}
template <int N>
__device__ __forceinline__ float row_value(float v) {
    const int q = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(q, q, 0x150 + N, 0xf, 0xf, true));
}

// Lane l - N of every row of 16 lanes (cyclic).
template <int N>
__device__ __forceinline__ float row_rotated(float v) {
    const int q = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(q, q, 0x120 + N, 0xf, 0xf, true));
}

// x[i] += nl u_i and rt[i] += nrl u_i, u_i = row_value<N>(rt[i]), for four values: one multiply-add with
// a DPP operand each.  The leading s_nop covers the two wait
// states between a vector write of rt and its use as a DPP operand.
template <int N>
__device__ __forceinline__ void row_fmac4(double* x, double* rt, double nl, double nrl) {
    asm("s_nop 1\n\t"
        "v_fmac_f64_dpp %0, %4, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %5, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %2, %6, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %3, %7, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %4, %4, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %5, %5, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %6, %6, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %7, %7, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf"
        : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(rt[0]), "+v"(rt[1]), "+v"(rt[2]), "+v"(rt[3])
        : "v"(nl), "v"(nrl), "n"(N));
}
template <int N>
__device__ __forceinline__ void row_fmac4(float* x, float* rt, float nl, float nrl) {
    asm("s_nop 1\n\t"
        "v_fmac_f32_dpp %0, %4, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %5, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %6, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %7, %8 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %4, %4, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %5, %5, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %6, %6, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %7, %7, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf"
        : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]), "+v"(rt[0]), "+v"(rt[1]), "+v"(rt[2]), "+v"(rt[3])
        : "v"(nl), "v"(nrl), "n"(N));
}

// Steps of the candidates' chain in round 1, for one 16-column block (columns base + 0..15, a row per
// lane in x).  rt holds the block's 16 pivot rows in every row of 16 lanes (lane n: row base + n of the
// panel), so that a pivot row's value reaches all lanes as one DPP operand; reading it with v_readlane
// instead took 2.5 times as long.
template <typename T>
struct SpecChain {
    // factors the block: multipliers to x, rt and sl[k][lane]
    template <int K>
    static __device__ __forceinline__ void factor_step(T (&x)[16], T (&rt)[16], T (*sl)[64], int lane, int rel, int ln) {
        const T rinv = spec_recip(row_value<K>(rt[K]));
        const T l = rel > K ? x[K] * rinv : T(0);
        const T rl = ln > K ? rt[K] * rinv : T(0);
        x[K] = rel > K ? l : x[K];
        sl[K][lane] = l;
        constexpr int first = (K + 4) / 4 * 4;  // the next column group
#pragma unroll
        for (int kk = K + 1; kk < first; kk++) {
            const T u = row_value<K>(rt[kk]);
            rt[kk] -= rl * u;
            x[kk] -= l * u;
        }
#pragma unroll
        for (int kk = first; kk < 16; kk += 4) row_fmac4<K>(x + kk, rt + kk, -l, -rl);
    }
    // applies the block's step K (multipliers l, for the pivot rows rl) to another block
    template <int K>
    static __device__ __forceinline__ void apply_step(T (&x)[16], T (&rt)[16], T l, T rl) {
#pragma unroll
        for (int kk = 0; kk < 16; kk += 4) row_fmac4<K>(x + kk, rt + kk, -l, -rl);
    }
    // step P of X = U^{-1}, X U = I with a row of X per lane: s holds I - X_{<P} U so far, rt U's rows,
    // rd the reciprocals of its diagonal
    template <int P>
    static __device__ __forceinline__ void inverse_step(T (&s)[16], const T (&rt)[16], T rd) {
        s[P] *= row_value<P>(rd);
#pragma unroll
        for (int j = P + 1; j < 16; j++) s[j] -= s[P] * row_value<P>(rt[j]);
    }
    template <int... K>
    static __device__ __forceinline__ void factor(T (&x)[16], T (&rt)[16], T (*sl)[64], int lane, int rel, int ln,
                                                  std::integer_sequence<int, K...>) {
        (factor_step<K>(x, rt, sl, lane, rel, ln), ...);
    }
    template <int... K>
    static __device__ __forceinline__ void apply(T (&x)[16], T (&rt)[16], const T (*sl)[64], int lane, int pl,
                                                 std::integer_sequence<int, K...>) {
        (apply_step<K>(x, rt, sl[K][lane], sl[K][pl]), ...);
    }
    template <int... P>
    static __device__ __forceinline__ void inverse(T (&s)[16], const T (&rt)[16], T rd,
                                                   std::integer_sequence<int, P...>) {
        (inverse_step<P>(s, rt, rd), ...);
    }
};

// Row ln of |X| |U| summed (X = U^{-1}, a row of each per lane, in every row of 16 lanes): what an explicit
// inverse multiplies the rounding of the product by.
template <typename T, int... J>
__device__ __forceinline__ T spec_condition(const T (&x)[16], const T (&u)[16], int ln, std::integer_sequence<int, J...>) {
    T rows = T(0), sum = T(0);
#pragma unroll
    for (int i = 0; i < 16; i++) rows += i >= ln ? (T)fabs(u[i]) : T(0);
    ((sum += (T)fabs(x[J]) * row_value<J>(rows)), ...);
    return sum;
}
// Largest such sum of a panel that may stand: the correction below leaves (eps cond)^2 of it, which is below
// eps up to here.  Wings stay far below (elliptic 12 x 100: 350, 64 x 64: 35).
__device__ __forceinline__ double spec_condition_limit(double) { return 0x1p22; }
__device__ __forceinline__ float spec_condition_limit(float) { return 0x1p9f; }

// R rows per lane: 64 R candidates.  Grid (x: shares of the rows, z: matrices), 256 threads.
template <typename T, int R>
__global__ __launch_bounds__(256) void k_panel_spec(T* __restrict__ a, int64_t lda, int n, int k0, int kb,
                                                    int32_t* __restrict__ ipiv, int32_t* __restrict__ perm, int64_t sb,
                                                    SpecBufs<T> sp, int round) {
    using M = Mf16<T>;
    constexpr int KC = NB / 4;  // columns per wave: wave g holds columns [16 g, 16 g + 16)
    const int z = blockIdx.z, t = threadIdx.x, lane = t & 63;
    const int g = __builtin_amdgcn_readfirstlane(t >> 6);
    a += (int64_t)z * sb;
    if constexpr (R == 2) {
        const int stood = spec_stood(sp, z, round - 1);
        if (stood == round - 1) spec_commit(sp, z, a, lda, n, k0, kb, blockIdx.x * 256 + t, gridDim.x * 256);
        if (stood != 0) return;
    }
    int32_t* fail = sp.fail + (round - 1) * sp.batch + z;
    if (sp.keys && sp.ostate[z] >= kSpecFails) {
        if (blockIdx.x == 0 && t == 0) *fail = 1;
        return;
    }
    const int m = n - k0;
    __shared__ T sU[NB][NB + 1];     // the factored diagonal block, rows in pivot order, U negated
    __shared__ T sInv[4][16][17];    // inverses of U's 16 x 16 diagonal blocks
    __shared__ T s_l[2][KC][64 * R];  // multipliers of a column block
    __shared__ int s_pv[2][KC];      // its pivots
    __shared__ int s_row[64 * R];    // candidate -> row (relative to k0), -1: none
    __shared__ int s_pos[64 * R];    // candidate -> final row (candidates that became no pivot)
    __shared__ uint32_t s_cmap[R == 2 ? kSpecMaxRows / 32 : 1];  // rows that are candidates below the diagonal block
    __shared__ int s_bad, s_ill;
    // candidates: the diagonal rows, from round 2 on also rows of the earlier rounds' keys
    int crow = -1;  // row of candidate 64 + lane
    if constexpr (R == 2) {
        for (int e = t; e < (m + 31) / 32; e += 256) s_cmap[e] = 0u;
        // all other rows where they are that few; else round by round, lane = column: its worst row first, then its
        // other rows; entry e of the list sits in lane e
        int count = 0;
        if (!sp.keys && kb + lane < m) crow = kb + lane;
        for (int rd = 0; sp.keys && rd < round - 1; rd++) {
            const unsigned long long* keys = sp.keys + ((int64_t)(rd * sp.batch + z) * kSpecSlots) * NB + lane;
            unsigned long long key[kSpecSlots + 1];
            key[0] = 0ull;
#pragma unroll
            for (int s = 1; s <= kSpecSlots; s++) key[s] = keys[(s - 1) * NB];
#pragma unroll
            for (int s = 1; s <= kSpecSlots; s++) key[0] = key[s] > key[0] ? key[s] : key[0];
            // alike in every wave: the columns that round 1 found a row for (none where no row was checked)
            if (rd == 0 && (sp.fail[z] == 2 || __popcll(__ballot(key[0] != 0ull)) > kSpecMaxBroken)) {
                if (blockIdx.x == 0 && t == 0) *fail = 1;
                return;
            }
#pragma unroll
            for (int s = 0; s <= kSpecSlots; s++) {
                const int row = key[s] != 0ull ? (int)~(uint32_t)key[s] : -1;
                for (unsigned long long todo = __ballot(row >= kb && row < m); todo != 0ull && count < 64;
                     todo &= todo - 1) {
                    const int r = __builtin_amdgcn_readlane(row, __ffsll((long long)todo) - 1);
                    if (__ballot(crow == r) != 0ull) continue;
                    crow = lane == count ? r : crow;
                    count++;
                }
            }
        }
    }
    if (t < 64) {
        s_row[lane] = lane < kb ? lane : -1;
        if constexpr (R == 2) s_row[64 + lane] = crow;
        if (lane == 0) s_bad = s_ill = 0;
    }
    __syncthreads();
    if constexpr (R == 2)
        if (t < 64 && crow >= 0) atomicOr(&s_cmap[crow >> 5], 1u << (crow & 31));
    T x[R][KC];
    bool act[R];
    int step[R];  // column at which this row became the pivot
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int row = s_row[64 * q + lane];
        act[q] = row >= 0;
        step[q] = -1;
#pragma unroll
        for (int k = 0; k < KC; k++) {
            const int c = KC * g + k;
            x[q][k] = (act[q] && c < kb) ? a[(k0 + row) + (int64_t)(k0 + c) * lda]
                                         : (R == 1 && lane == c ? T(1) : T(0));  // round 1: identity beyond kb
        }
    }
    // the wave's first 16 other rows, in flight while the candidates are factored: lane l holds row
    // l % 16, columns M::k(l, r) of each 16-block
    const int tiles = (m - kb + 15) / 16, ln = lane & 15;
    typename M::vacc y[4];
    auto load_rows = [&](int tile) {
        const int row = kb + 16 * tile + ln;
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                y[b][r] = (tile < tiles && row < m)
                              ? a[(k0 + row) + (int64_t)(k0 + 16 * b + M::k(lane, r)) * lda]
                              : T(0);
    };
    // with more than one work-group, the first writes the candidates' result instead
    const int share = gridDim.x > 1 ? (int)blockIdx.x - 1 : 0, shares = gridDim.x > 1 ? gridDim.x - 1 : 1;
    if (share >= 0) load_rows(4 * share + g);
    // where the rows are as the interchanges go on: src = candidate now at position `lane`, oval =
    // candidate now at the place of candidate 64 + lane; pp = the position pivot `lane` came from
    int src = lane, oval = 64 + lane, pp = lane;
    bool bad = false, over1 = false;
    // candidate p becomes the pivot of column j
    auto take = [&](int j, int p) {
        if constexpr (R == 2) {
            const int did = __builtin_amdgcn_readlane(src, j);
            if (p != did) {  // position j's row and p change places
                const unsigned long long in = __ballot(src == p);
                if (in != 0ull) {
                    const int jj = __ffsll((long long)in) - 1;
                    pp = lane == j ? jj : pp;
                    src = lane == j ? p : (lane == jj ? did : src);
                } else {
                    const int e = (__ffsll((long long)__ballot(oval == p)) - 1) & 63;
                    const int place = __builtin_amdgcn_readlane(crow, e);
                    pp = lane == j ? place : pp;
                    src = lane == j ? p : src;
                    oval = lane == e ? did : oval;
                }
            }
        }
#pragma unroll
        for (int q = 0; q < R; q++)
            if (64 * q + lane == p) {
                act[q] = false;
                step[q] = j;
            }
    };
    if constexpr (R == 1) {
        constexpr auto k16 = std::make_integer_sequence<int, KC>{};
#pragma unroll 1
        for (int b = 0; b < 4; b++) {
            const int buf = b & 1, pl = KC * b + ln;  // lane of the block's pivot row ln
            if (g >= b) {
                // this wave's columns in the block's pivot rows, for every row of 16 lanes
                T rt[KC];
                if (g == b) {  // factor the block; the waves right of it apply it after the barrier
#pragma unroll
                    for (int k = 0; k < KC; k++) rt[k] = __shfl(x[0][k], pl);
                    SpecChain<T>::factor(x[0], rt, s_l[buf], lane, lane - KC * b, ln, k16);
                }
                lds_sync();
                if (g > b) {
#pragma unroll
                    for (int k = 0; k < KC; k++) rt[k] = __shfl(x[0][k], pl);
                    SpecChain<T>::apply(x[0], rt, s_l[buf], lane, pl, k16);
                }
            } else {
                lds_sync();
            }
        }
        step[0] = lane;
    } else {
#pragma unroll 1
        for (int b = 0; b < 4; b++) {
            if (KC * b >= kb) break;
            const int buf = b & 1;
            if (g == b) {
#pragma unroll
                for (int k = 0; k < KC; k++) {
                    const int j = KC * b + k;
                    if (j < kb) {
                        const int did = __builtin_amdgcn_readlane(src, j);  // the row at position j
                        T v[R];
#pragma unroll
                        for (int q = 0; q < R; q++) v[q] = act[q] ? (T)fabs(x[q][k]) : T(-1);
                        const T dv = did >= 64 ? lane_value(v[R - 1], did & 63) : lane_value(v[0], did);
                        int p = did;
                        if (__ballot(v[0] > dv || v[R - 1] > dv) != 0ull) {
                            T best = v[0];
                            int bi = lane;
                            argmax_merge(best, bi, v[R - 1], 64 + lane);
                            wave_argmax(best, bi);
                            p = bi;
                            bad = bad || __popcll(__ballot(v[0] == best)) + __popcll(__ballot(v[R - 1] == best)) != 1;
                        }
                        take(j, p);
                        // xr: the pivot's row among the lane's R rows
                        auto eliminate = [&](T (&xr)[KC]) {
                            const T rinv = spec_recip(lane_value(xr[k], p & 63));
                            T l[R];
#pragma unroll
                            for (int q = 0; q < R; q++) {
                                l[q] = act[q] ? x[q][k] * rinv : T(0);
                                x[q][k] = act[q] ? l[q] : x[q][k];
                                s_l[buf][k][64 * q + lane] = l[q];
                            }
                            if (lane == 0) s_pv[buf][k] = p;
                            T u[KC];
#pragma unroll
                            for (int kk = k + 1; kk < KC; kk++) u[kk] = lane_value(xr[kk], p & 63);
#pragma unroll
                            for (int kk = k + 1; kk < KC; kk++)
#pragma unroll
                                for (int q = 0; q < R; q++) x[q][kk] -= l[q] * u[kk];
                        };
                        if (p < 64)
                            eliminate(x[0]);
                        else
                            eliminate(x[R - 1]);
                    }
                }
            }
            lds_sync();
            if (g != b) {
                const int kn = min(KC, kb - KC * b);
                int pn = __builtin_amdgcn_readfirstlane(s_pv[buf][0]);
                T lnx[R];
#pragma unroll
                for (int q = 0; q < R; q++) lnx[q] = s_l[buf][0][64 * q + lane];
                for (int k = 0; k < kn; k++) {
                    const int p = pn, kx = k + 1 < kn ? k + 1 : k;
                    T l[R];
#pragma unroll
                    for (int q = 0; q < R; q++) {
                        l[q] = lnx[q];
                        lnx[q] = s_l[buf][kx][64 * q + lane];
                    }
                    const int pv = s_pv[buf][kx];
                    take(KC * b + k, p);
                    if (g > b) {
                        T u[KC];
                        if (p < 64) {
#pragma unroll
                            for (int kk = 0; kk < KC; kk++) u[kk] = lane_value(x[0][kk], p & 63);
                        } else {
#pragma unroll
                            for (int kk = 0; kk < KC; kk++) u[kk] = lane_value(x[R - 1][kk], p & 63);
                        }
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int kk = 0; kk < KC; kk++)
#pragma unroll
                            for (int q = 0; q < R; q++) x[q][kk] -= l[q] * u[kk];
                    }
                    pn = __builtin_amdgcn_readfirstlane(pv);
                }
            }
        }
    }
    // every multiplier of the candidates (columns before a row's own pivot) is below 1 (rounds 2 and 3, which
    // searched the pivot among them: at most 1)
    constexpr T strict = T(1) - T(64) * (sizeof(T) == 8 ? (T)2.2e-16 : (T)1.2e-7f);
#pragma unroll
    for (int q = 0; q < R; q++)
#pragma unroll
        for (int k = 0; k < KC; k++) {
            const int c = KC * g + k;
            const bool mult = (R == 1 ? step[q] > c : act[q] || step[q] > c) && c < kb;
            over1 = over1 || (mult && !(fabs(x[q][k]) <= (R == 1 ? strict : T(1))));
        }
    // round 1 goes on to the other rows after such an |l| among the candidates (they are all
    // candidates again, the keys of the others are wanted)
    if (R == 1 && blockIdx.x == 0 && __ballot(over1) != 0ull && lane == 0) atomicMax(fail, 1);
    bad = bad || (R == 2 && over1);
    if (__ballot(bad) != 0ull && lane == 0) s_bad = 1;
    // the diagonal block in pivot order (identity beyond kb), U negated for the products below
    if (R == 2 && kb < NB)
        for (int e = t; e < NB * NB; e += 256) {
            const int r = e & 63, c = e >> 6;
            if (r >= kb || c >= kb) sU[r][c] = r == c ? T(-1) : T(0);
        }
#pragma unroll
    for (int q = 0; q < R; q++)
        if (step[q] >= 0)
#pragma unroll
            for (int k = 0; k < KC; k++) {
                const int c = KC * g + k;
                if (R == 1 || c < kb) sU[step[q]][c] = c >= step[q] ? -x[q][k] : x[q][k];
            }
    if (g == 0) {
        s_pos[lane] = -1;
        if constexpr (R == 2) {
            s_pos[64 + lane] = -1;
            if (crow >= 0) s_pos[oval] = crow;
        }
    }
    __syncthreads();
    const bool badp = !spec_pivot_ok(sU[lane][lane]);
    if (s_bad != 0 || __ballot(badp) != 0ull) {
        if (blockIdx.x == 0 && t == 0) *fail = 1;
        // with a pivot that is not finite or zero the products below mean nothing
        return;
    }
    T* w = sp.w + (int64_t)z * sp.ldw * NB;
    if (blockIdx.x == 0) {
        for (int e = t; e < NB * kb; e += 256) {
            const int r = e % NB, c = e / NB;
            if (r < kb) w[r + (int64_t)c * sp.ldw] = c >= r ? -sU[r][c] : sU[r][c];
        }
#pragma unroll
        for (int q = 0; q < R; q++) {
            const int pos = s_pos[64 * q + lane];
            if (pos >= 0 && step[q] < 0)
#pragma unroll
                for (int k = 0; k < KC; k++)
                    if (KC * g + k < kb) w[pos + (int64_t)(KC * g + k) * sp.ldw] = x[q][k];
        }
        if (g == 0) {
            if (lane < kb) ipiv[(int64_t)z * n + k0 + lane] = k0 + pp + 1;
            // composed interchanges (destination, source), as wave_compose_swaps lists them
            int32_t* out = perm + (int64_t)z * kPermInts;
            const bool in_pair = lane < kb && src != lane;
            const bool out_pair = R == 2 && crow >= 0 && oval != 64 + lane;
            const unsigned long long mi = __ballot(in_pair), mo = __ballot(out_pair);
            const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
            const int ni = __popcll(mi);
            if (in_pair) {
                const int e = __popcll(mi & below);
                out[1 + 2 * e] = k0 + lane;
                out[2 + 2 * e] = k0 + s_row[src];
            }
            if (out_pair) {
                const int e = ni + __popcll(mo & below);
                out[1 + 2 * e] = k0 + crow;
                out[2 + 2 * e] = k0 + s_row[oval];
            }
            if (lane == 0) out[0] = ni + __popcll(mo);
        }
    }
    if (m <= kb || share < 0 || (R == 2 && !sp.keys)) return;
    // inverse of U's diagonal block g, a row per lane (in every row of 16 lanes)
    {
        T rt[16], s[16];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            rt[i] = -sU[16 * g + ln][16 * g + i];  // (the multipliers below the diagonal are not read)
            s[i] = i == ln ? T(1) : T(0);
        }
        const T rd = T(-1) / sU[16 * g + ln][16 * g + ln];
        SpecChain<T>::inverse(s, rt, rd, std::make_integer_sequence<int, 16>{});
        if (lane < 16)
#pragma unroll
            for (int i = 0; i < 16; i++) sInv[g][ln][i] = s[i];
        const T cond = spec_condition(s, rt, ln, std::make_integer_sequence<int, 16>{});
        if (__ballot(!(cond <= spec_condition_limit(T(0)))) != 0ull && lane == 0) s_ill = 1;
    }
    __syncthreads();
    if (s_ill != 0) {  // the rows' multipliers would not be accurate
        if (t == 0) atomicMax(fail, 2);
        return;
    }
    // the other rows, 16 per wave and step
    bool failed = false;
    for (int tile = 4 * share + g; tile < tiles; tile += 4 * shares) {
        if (tile >= 4 * shares) load_rows(tile);  // the first tile is here already
        const int row = kb + 16 * tile + ln;
        bool use = row < m;
        if constexpr (R == 2) use = use && ((s_cmap[row >> 5] >> (row & 31)) & 1u) == 0u;
#pragma unroll
        for (int b = 0; b < 4; b++) {
#pragma unroll
            for (int c = 0; c < b; c++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    y[b] = M::mfma(sU[16 * c + M::k(lane, r)][16 * b + ln], y[c][r], y[b]);
            typename M::vacc s = {T(0), T(0), T(0), T(0)};
#pragma unroll
            for (int r = 0; r < 4; r++) s = M::mfma(sInv[b][M::k(lane, r)][ln], y[b][r], s);
            // s += Uinv_bb^T (y_b - U_bb^T s)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int k = M::k(lane, r);
                y[b] = M::mfma(k <= ln ? sU[16 * b + k][16 * b + ln] : T(0), s[r], y[b]);
            }
#pragma unroll
            for (int r = 0; r < 4; r++) s = M::mfma(sInv[b][M::k(lane, r)][ln], y[b][r], s);
            y[b] = s;
        }
        bool over = false;
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                over = over || !((T)fabs(y[b][r]) <= strict);
                if (use) w[row + (int64_t)(16 * b + M::k(lane, r)) * sp.ldw] = y[b][r];
            }
        over = over && use;
        if (__ballot(over) != 0ull) {
            failed = true;
            if (sp.keys && round < kSpecRounds) {  // per column the row of the largest |l| among the wave's 16
#pragma unroll
                for (int b = 0; b < 4; b++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const T v = use ? (T)fabs(y[b][r]) : T(0);
                        const float f = v <= strict ? 0.0f : (v < T(3e38) ? (float)v : 3.4e38f);
                        float top = fmaxf(f, row_rotated<8>(f));
                        top = fmaxf(top, row_rotated<4>(top));
                        top = fmaxf(top, row_rotated<2>(top));
                        top = fmaxf(top, row_rotated<1>(top));
                        const bool hit = f > 0.0f && f == top;
                        const uint32_t first = (uint32_t)(__ballot(hit) >> (lane & 48)) & ((1u << ln) - 1u);
                        if (hit && first == 0u)
                            atomicMax(&sp.keys[((int64_t)((round - 1) * sp.batch + z) * kSpecSlots + tile % kSpecSlots) *
                                                   NB +
                                               16 * b + M::k(lane, r)],
                                      ((unsigned long long)__float_as_uint(f) << 32) | (uint32_t)~row);
                    }
            }
        }
    }
    if (failed && lane == 0) *fail = 1;
}

template <typename T, int NT, int Q, int IB>
__global__ __launch_bounds__(NT) void k_panel_reg(T* __restrict__ a, int64_t lda, int n, int k0, int kb,
                                                  int32_t* __restrict__ ipiv, int32_t* __restrict__ info,
                                                  int32_t* __restrict__ perm, int64_t sb, SpecBufs<T> sp) {
    constexpr int NW = NT / 64;
    a += (int64_t)blockIdx.z * sb;  // batch: one matrix per blockIdx.z
    // after a speculative panel: nothing to do where one of its earlier rounds stood; where the last did,
    // the launch's work-groups copy its result; work-group 0 factors the panel where all failed
    if (sp.on && spec_settled(sp, blockIdx.z, blockIdx.x == 0 && threadIdx.x == 0)) {
        if (spec_stood(sp, blockIdx.z, sp.rounds - 1) == 0)
            spec_commit(sp, blockIdx.z, a, lda, n, k0, kb, blockIdx.x * NT + threadIdx.x, gridDim.x * NT);
        return;
    }
    if (blockIdx.x != 0) return;
    ipiv += (int64_t)blockIdx.z * n;
    info += blockIdx.z;
    perm += (int64_t)blockIdx.z * kPermInts;
    __shared__ T s_val[NW];
    __shared__ int s_idx[NW];
    __shared__ T s_rowp[IB], s_rowc[IB];
    __shared__ T s_inv[NB / IB][IB][IB];
    __shared__ T s_blk[IB][IB];
    __shared__ T s_u[IB][IB];
    __shared__ int s_arg[NB], s_piv[NB];
    __shared__ int s_pd[2 * NB], s_ps[2 * NB], s_pcnt, s_zero;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    if (t == 0) s_zero = 0;
    T x[Q][IB];

    for (int c0 = k0, s = 0; c0 < k0 + kb; c0 += IB, s++) {
        const int ib = min(IB, k0 + kb - c0);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int r = k0 + t + NT * q;
#pragma unroll
            for (int j = 0; j < IB; j++) x[q][j] = (r < n && j < ib) ? a[r + (int64_t)(c0 + j) * lda] : T(0);
        }
        // updates from the earlier sub-panels sp < s (rows b0 .. b0+IB of block sp hold U after this);
        // when registers allow, the L block of round sp + 1 is loaded while round sp computes (two
        // register buffers, rounds taken in pairs so that both stay statically indexed)
        T l0[Q][IB], l1[Q][IB];
        auto load_l = [&](T (&l)[Q][IB], int b) {
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const int r = k0 + t + NT * q;
#pragma unroll
                for (int p = 0; p < IB; p++) l[q][p] = (r >= b + IB && r < n) ? a[r + (int64_t)(b + p) * lda] : T(0);
            }
        };
        auto round = [&](int sp, T (&lc)[Q][IB], T (&ln)[Q][IB], bool prefetch) {
            const int b0 = k0 + sp * IB;
            if (prefetch && sp + 1 < s) load_l(ln, b0 + IB);
            const int jj = t - (b0 - k0);  // owners of the block's rows: q = 0
            if (jj >= 0 && jj < IB) {
#pragma unroll
                for (int j = 0; j < IB; j++) s_blk[jj][j] = x[0][j];
            }
            lds_sync();
            if (t < IB * IB) {
                const int i = t / IB, j = t % IB;
                T u = T(0);
                for (int p = 0; p <= i; p++) u += s_inv[sp][i][p] * s_blk[p][j];
                s_u[i][j] = u;
            }
            lds_sync();
            if (jj >= 0 && jj < IB) {
#pragma unroll
                for (int j = 0; j < IB; j++) x[0][j] = s_u[jj][j];
            }
#pragma unroll
            for (int q = 0; q < Q; q++) {
                const int r = k0 + t + NT * q;
                if (r >= b0 + IB && r < n) {
#pragma unroll
                    for (int j = 0; j < IB; j++) {
                        T acc = x[q][j];
#pragma unroll
                        for (int p = 0; p < IB; p++) acc -= lc[q][p] * s_u[p][j];
                        x[q][j] = acc;
                    }
                }
            }
            lds_sync();  // s_u, s_blk reused by the next block
        };
        if constexpr (Q * IB * sizeof(T) <= 256) {
            if (s > 0) load_l(l0, k0);
            for (int sp = 0; sp < s; sp += 2) {
                round(sp, l0, l1, true);
                if (sp + 1 < s) round(sp + 1, l1, l0, true);
            }
        } else {  // registers for one buffer only: each round loads its own block first
            for (int sp = 0; sp < s; sp++) {
                load_l(l0, k0 + sp * IB);
                round(sp, l0, l1, false);
            }
        }
        // factor the sub-panel
#pragma unroll
        for (int jj = 0; jj < IB; jj++) {
            if (jj < ib) {
                const int c = c0 + jj;
                T best = T(-1);
                int bi = n;
#pragma unroll
                for (int q = 0; q < Q; q++) {
                    const int r = k0 + t + NT * q;
                    if (r >= c && r < n) argmax_merge(best, bi, (T)fabs(x[q][jj]), r);
                }
                wave_argmax(best, bi);
                if (lane == 0) {
                    s_val[w] = best;
                    s_idx[w] = bi;
                }
                lds_sync();
                best = s_val[0];
                bi = s_idx[0];
#pragma unroll
                for (int ww = 1; ww < NW; ww++) argmax_merge(best, bi, s_val[ww], s_idx[ww]);
                // a column of NaNs wins no comparison and leaves bi = n: take row c then (LAPACK's
                // idamax also stays on the first entry), so every row index below stays in [c, n)
                const int p = (bi >= c && bi < n) ? bi : c;
                const int tp = (p - k0) % NT, qp = (p - k0) / NT;
                const int tc = (c - k0) % NT, qc = (c - k0) / NT;
                if (t == tp) {
#pragma unroll
                    for (int q = 0; q < Q; q++)
                        if (q == qp) {
#pragma unroll
                            for (int j = 0; j < IB; j++) s_rowp[j] = x[q][j];
                        }
                }
                if (t == tc) {
#pragma unroll
                    for (int q = 0; q < Q; q++)
                        if (q == qc) {
#pragma unroll
                            for (int j = 0; j < IB; j++) s_rowc[j] = x[q][j];
                        }
                }
                lds_sync();
                const T piv = s_rowp[jj];
                const bool nz = piv != T(0);
                if (t == 0) {
                    s_arg[c - k0] = p;
                    s_piv[c - k0] = nz ? p : c;
                    if (!nz && s_zero == 0) s_zero = c + 1;
                }
                if (nz) {
                    if (p != c) {
                        if (t == tc) {
#pragma unroll
                            for (int q = 0; q < Q; q++)
                                if (q == qc) {
#pragma unroll
                                    for (int j = 0; j < IB; j++) x[q][j] = s_rowp[j];
                                }
                        }
                        if (t == tp) {
#pragma unroll
                            for (int q = 0; q < Q; q++)
                                if (q == qp) {
#pragma unroll
                                    for (int j = 0; j < IB; j++) x[q][j] = s_rowc[j];
                                }
                        }
                    }
                    const T rinv = T(1) / piv;
#pragma unroll
                    for (int q = 0; q < Q; q++) {
                        const int r = k0 + t + NT * q;
                        if (r > c && r < n) {
                            const T l = x[q][jj] * rinv;
                            x[q][jj] = l;
#pragma unroll
                            for (int j = jj + 1; j < IB; j++) x[q][j] -= l * s_rowp[j];
                        }
                    }
                }
                lds_sync();  // s_rowp / s_rowc / s_val reused by the next column
            }
        }
        // sub-panel back to memory
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int r = k0 + t + NT * q;
            if (r < n) {
#pragma unroll
                for (int j = 0; j < IB; j++)
                    if (j < ib) a[r + (int64_t)(c0 + j) * lda] = x[q][j];
            }
        }
        // the sub-panel's interchanges on the panel's other columns, as one gather / scatter
        if (t < 64) {
            const int np = wave_compose_swaps(c0, ib, s_piv + (c0 - k0), s_pd, s_ps);
            if (t == 0) s_pcnt = np;
        }
        __syncthreads();
        {
            // whole columns per pass: every source of a column is read before any of its rows is written
            const int pairs = s_pcnt;
            if (pairs > 0) {
                const int cpi = NT / pairs, cl = t / pairs, pr = t % pairs;
                for (int cb = 0; cb < kb; cb += cpi) {
                    const int col = k0 + cb + cl;
                    const bool act = cl < cpi && cb + cl < kb && (col < c0 || col >= c0 + ib);
                    T v = T(0);
                    if (act) v = a[s_ps[pr] + (int64_t)col * lda];
                    __syncthreads();
                    if (act) a[s_pd[pr] + (int64_t)col * lda] = v;
                    __syncthreads();
                }
            }
        }
        // inverse of the unit-lower diagonal block, for the later sub-panels
        if (c0 + ib < k0 + kb) {
            const int jj = t - (c0 - k0);
            if (jj >= 0 && jj < IB) {
#pragma unroll
                for (int j = 0; j < IB; j++) s_blk[jj][j] = x[0][j];
            }
            lds_sync();
            if (t < IB) {
                const int j = t;
                T col[IB];
#pragma unroll
                for (int i = 0; i < IB; i++) col[i] = i == j ? T(1) : T(0);
#pragma unroll
                for (int i = 0; i < IB; i++) {
                    if (i > j) {
                        T v = T(0);
#pragma unroll
                        for (int p = 0; p < IB; p++)
                            if (p >= j && p < i) v -= s_blk[i][p] * col[p];
                        col[i] = v;
                    }
                }
#pragma unroll
                for (int i = 0; i < IB; i++) s_inv[s][i][j] = col[i];
            }
        }
        __syncthreads();
    }
    // pivots, first zero pivot, and the panel's composed interchanges for the rest of the matrix
    if (t < kb) ipiv[k0 + t] = s_arg[t] + 1;
    if (t == 0 && s_zero != 0 && info[0] == 0) info[0] = s_zero;
    if (t < 64) {
        const int np = wave_compose_swaps(k0, kb, s_piv, s_pd, s_ps);
        if (t == 0) s_pcnt = np;
    }
    __syncthreads();
    const int np = s_pcnt;
    for (int e = t; e < np; e += NT) {
        perm[1 + 2 * e] = s_pd[e];
        perm[2 + 2 * e] = s_ps[e];
    }
    if (t == 0) perm[0] = np;
}

// ---- cooperative tall panel ---------------------------------------------------------------------
// k_panel_coop: G work-groups of NT threads factor the panel rows [k0, n) x columns [k0, k0 + kb)
// together (kb <= NB).  Thread t of group g owns row k0 + g NT + t; the group keeps its NT rows of
// the panel in LDS, column-major (consecutive threads, consecutive banks), from the first column to
// the last.  Per column, one exchange through global memory: the first wave of every group
// publishes the group's local pivot candidate (|value|, row) and that row's values (group 0 also
// the diagonal row) from LDS, releases once, and counts the group in at a per-column counter (one
// atomic add each, then a bounded spin).  Every group then
// picks the same pivot (largest |value|, first row on ties: LAPACK's choice), the owners of the
// pivot and diagonal rows exchange them, and each group scales and updates its own rows.  Exchange
// buffers (per matrix): cval / crow [NB][kCoopMaxGroups], xrow [NB][kCoopMaxGroups + 1][NB] (slot
// kCoopMaxGroups: the diagonal row), counters ctr [NB], zeroed before the launch.  A spin that runs
// out (the groups were not all resident), or a pivot row outside [c, n) read back from the exchange,
// leaves info = kCoopStalled instead of waiting for ever or indexing out of bounds.
// Group 0 writes ipiv and the panel's composed interchanges for k_swap_trsm, as k_panel_reg does.
//
// After a speculative panel (k_panel_spec) it factors only the matrices for which all rounds failed;
// where the last round stood, the groups copy its result into the matrix instead.
constexpr int kCoopMaxGroups = 64;   // work-groups of one launch; all of them must be resident at once
constexpr int kCoopMinRows = 1024;   // shorter panels stay in one work-group (k_panel_reg)
constexpr unsigned kCoopSpinLimit = 1u << 22;  // default bound of every wait (tvlm_lu_set_coop_spin_limit)
constexpr int kCoopStalled = -999;
constexpr int kCoopCtr = NB + 4;  // ints between the counter sets of a panel and matrix (NB counters each)
constexpr int64_t kCoopXrow = (int64_t)NB * (kCoopMaxGroups + 1) * NB;  // xrow per matrix

template <typename T>
__device__ __forceinline__ void st_agent(T* p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ T ld_agent(T* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// threads (= rows) per cooperative work-group: NT rows x NB columns of T = 128 KB of LDS
template <typename T>
constexpr int coop_threads() {
    return sizeof(T) == 4 ? 512 : 256;
}

template <typename T, int NT>
__global__ __launch_bounds__(NT) void k_panel_coop(T* __restrict__ a, int64_t lda, int n, int k0, int kb, int G,
                                                   int32_t* __restrict__ ipiv, int32_t* __restrict__ info,
                                                   int32_t* __restrict__ perm, int64_t sb, int32_t* ctr, T* cval,
                                                   int32_t* crow, T* xrow, unsigned spin_limit, int32_t* fail,
                                                   SpecBufs<T> sp) {
    constexpr int NW = NT / 64, MG = kCoopMaxGroups;
    const int z = blockIdx.z, g = blockIdx.x, t = threadIdx.x, lane = t & 63, w = t >> 6;
    if (sp.on && spec_settled(sp, z, g == 0 && t == 0)) {
        if (spec_stood(sp, z, sp.rounds - 1) == 0)
            spec_commit(sp, z, a + (int64_t)z * sb, lda, n, k0, kb, g * NT + t, G * NT);
        return;
    }
    a += (int64_t)z * sb;
    ipiv += (int64_t)z * n;
    info += z;
    perm += (int64_t)z * kPermInts;
    ctr += (int64_t)z * kCoopCtr;
    cval += (int64_t)z * NB * MG;
    crow += (int64_t)z * NB * MG;
    xrow += (int64_t)z * kCoopXrow;
    const int m = n - k0, i = g * NT + t;  // this thread's row: k0 + i
    const bool mine = i < m;
    extern __shared__ unsigned char coop_lds[];
    T* xs = reinterpret_cast<T*>(coop_lds);  // xs[jj * NT + t]: column jj of this group's row t
    __shared__ T s_val[NW];
    __shared__ int s_idx[NW];
    __shared__ T s_prow[NB], s_crow[NB];
    __shared__ int s_p, s_fail, s_zero, s_arg[NB], s_piv[NB];
    __shared__ int s_pd[2 * NB], s_ps[2 * NB], s_pcnt;
    if (t == 0) {
        s_fail = 0;
        s_zero = 0;
    }
    for (int jj = 0; jj < kb; jj++) xs[jj * NT + t] = mine ? a[k0 + i + (int64_t)(k0 + jj) * lda] : T(0);
    __syncthreads();
    for (int j = 0; j < kb; j++) {
        const int c = k0 + j;
        // this group's candidate: largest |a(r, c)| over its rows r >= c, first row on ties
        T best = T(-1);
        int bi = n;
        if (mine && i >= j) {
            best = (T)fabs(xs[j * NT + t]);
            bi = k0 + i;
        }
        wave_argmax(best, bi);
        if (lane == 0) {
            s_val[w] = best;
            s_idx[w] = bi;
        }
        __syncthreads();
        best = s_val[0];
        bi = s_idx[0];
#pragma unroll
        for (int ww = 1; ww < NW; ww++) argmax_merge(best, bi, s_val[ww], s_idx[ww]);
        // publish and meet: wave 0 writes this group's candidate row and (group 0) the diagonal row
        // straight from LDS, then the candidate, releases once, and its lane 0 counts the group in
        // and waits for the others; the other waves go straight to the barrier
        T* xr = xrow + (int64_t)j * (MG + 1) * NB;
        if (w == 0) {
            if (bi < n && lane < kb) st_agent(&xr[g * NB + lane], xs[lane * NT + (bi - k0 - g * NT)]);
            if (g == 0 && lane < kb) st_agent(&xr[MG * NB + lane], xs[lane * NT + j]);  // row c: local row j
            if (lane == 0) {
                st_agent(&cval[j * MG + g], best);
                st_agent(&crow[j * MG + g], bi);
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
            if (lane == 0) {
                __hip_atomic_fetch_add(&ctr[j], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                unsigned spins = 0;
                while (__hip_atomic_load(&ctr[j], __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT) < G) {
                    if (++spins > spin_limit) {
                        s_fail = 1;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
            }
        }
        __syncthreads();
        // the pivot: the same reduction in every group
        if (w == 0) {
            T v = T(-1);
            int ri = n;
            if (lane < G) {
                v = ld_agent(&cval[j * MG + lane]);
                ri = ld_agent(&crow[j * MG + lane]);
            }
            wave_argmax(v, ri);
            if (lane == 0) {
                // ri == n: no group had a candidate (a column of NaNs): row c, as LAPACK's idamax;
                // any other pivot row outside [c, n) can only come from a failed exchange: keep every
                // index below in bounds and report it
                const bool ok = ri >= c && ri < n;
                s_p = ok ? ri : c;
                if (!ok && ri != n) s_fail = 1;
            }
        }
        __syncthreads();
        const int p = s_p;
        const int gw = (p - k0) / NT;
        if (t < kb) s_prow[t] = ld_agent(&xr[gw * NB + t]);
        if (t >= 64 && t - 64 < kb) s_crow[t - 64] = ld_agent(&xr[MG * NB + (t - 64)]);
        __syncthreads();
        const T piv = s_prow[j];
        const bool nz = piv != T(0);
        if (g == 0 && t == 0) {
            s_arg[j] = p;
            s_piv[j] = nz ? p : c;
            if (!nz && s_zero == 0) s_zero = c + 1;
        }
        if (nz) {
            if (p != c) {
                if (g == 0 && t < kb) xs[t * NT + j] = s_prow[t];
                if (gw == g && t < kb) xs[t * NT + (p - k0 - g * NT)] = s_crow[t];
                __syncthreads();
            }
            if (mine && i > j) {
                const T l = xs[j * NT + t] * (T(1) / piv);
                xs[j * NT + t] = l;
#pragma unroll 8
                for (int jj = j + 1; jj < kb; jj++) xs[jj * NT + t] -= l * s_prow[jj];
            }
        }
        __syncthreads();  // s_val / s_prow / s_crow / s_p reused by the next column
    }
    if (mine)
        for (int jj = 0; jj < kb; jj++) a[k0 + i + (int64_t)(k0 + jj) * lda] = xs[jj * NT + t];
    // any group whose wait ran out marks the matrix (k_coop_fail_info turns the mark into info)
    if (t == 0 && s_fail) __hip_atomic_fetch_or(&fail[z], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (g != 0) return;
    if (t < kb) ipiv[k0 + t] = s_arg[t] + 1;
    if (t == 0) {
        if (s_fail)
            info[0] = kCoopStalled;
        else if (s_zero != 0 && info[0] == 0)
            info[0] = s_zero;
    }
    if (t < 64) {
        const int np = wave_compose_swaps(k0, kb, s_piv, s_pd, s_ps);
        if (t == 0) s_pcnt = np;
    }
    __syncthreads();
    const int np = s_pcnt;
    for (int e = t; e < np; e += NT) {
        perm[1 + 2 * e] = s_pd[e];
        perm[2 + 2 * e] = s_ps[e];
    }
    if (t == 0) perm[0] = np;
}

// Row interchanges of one panel on the columns outside it, then for the columns right of the panel
// U12 = L11^{-1} A12 (L11 unit lower).  A wave takes 16 columns, which no other wave touches: every
// value it needs is read before any is written, so the waves meet only once, for L11.  U12 is formed
// on the matrix cores, 16 rows at a time: Z_b = Linv_bb (A_b - sum_{c<b} L_bc Z_c), Linv_bb the
// inverse of L11's 16 x 16 diagonal block (each work-group inverts the four, a wave each), corrected once
// with its residual (multipliers of up to 1 allow entries of 2^14 in that inverse; without the correction
// |A12 - L11 U12| reached 1400 eps |L11| |U12|, with it as little as by substitution); the MFMA
// output layout is the second operand's, so the blocks chain in registers, and the block's rows are
// read through the interchanges and written once.
// Bound by the latency of the scattered column reads: 15.4 us per launch (mean over a factorisation of
// N = 4096, FP64) against 60.7 us for forward substitution of a 64 x 64 block in LDS, one row per step.
// mode: 0 = interchanges on both sides and U12 on the right; 1 = interchanges only; 2 = U12 only
// (the right blocks, no interchanges).  With gtab, the left blocks before column left0 take the
// interchanges into their gather lists instead of their columns (deferred interchanges, below).  The
// left blocks start at column lbase, the right ones at rbase (default: right after the panel).
template <typename T>
__global__ __launch_bounds__(256) void k_swap_trsm(T* __restrict__ a, int64_t lda, int n, int k0, int kb, int nleft,
                                                   const int32_t* __restrict__ perm, int64_t sb, int mode = 0,
                                                   int left0 = 0, int32_t* __restrict__ gtab = nullptr, int lbase = 0,
                                                   int rbase = -1) {
    using M = Mf16<T>;
    a += (int64_t)blockIdx.z * sb;
    perm += (int64_t)blockIdx.z * kPermInts;
    __shared__ int s_pd[2 * NB], s_ps[2 * NB];
    __shared__ int s_map[NB];        // row of the block -> the row it comes from
    __shared__ T s_l[NB][NB + 1];    // -L11 below the diagonal
    __shared__ T s_inv[4][16][17];   // inverses of its 16 x 16 diagonal blocks
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const bool left = (int)blockIdx.x < nleft;
    const int col0 = left ? lbase + blockIdx.x * 64 : (rbase < 0 ? k0 + kb : rbase) + (blockIdx.x - nleft) * 64;
    const int colend = left ? k0 : n;
    const int cnt = mode == 2 ? 0 : perm[0];
    if (left && gtab && col0 < left0) {
        // g'[dst] = g[src] for every pair of the panel's composed interchanges (cnt <= 2 NB)
        int32_t* g = gtab + ((int64_t)blockIdx.z * ((n + NB - 1) / NB) + col0 / NB) * n;
        const int v = t < cnt ? g[perm[2 + 2 * t]] : 0;
        __syncthreads();
        if (t < cnt) g[perm[1 + 2 * t]] = v;
        return;
    }
    const bool solve = !left && mode != 1;
    if (cnt == 0 && !solve) return;
    for (int e = t; e < cnt; e += 256) {
        s_pd[e] = perm[1 + 2 * e];
        s_ps[e] = perm[2 + 2 * e];
    }
    if (t < NB) s_map[t] = k0 + t;
    if (solve)
        for (int e = t; e < NB * NB; e += 256) {
            const int r = e & 63, c = e >> 6;
            s_l[r][c] = (r < kb && c < r) ? -a[(k0 + r) + (int64_t)(k0 + c) * lda] : T(0);
        }
    __syncthreads();
    if (solve) {
        if (t < cnt && s_pd[t] >= k0 && s_pd[t] < k0 + kb) s_map[s_pd[t] - k0] = s_ps[t];
        // unit lower: X_ij = delta_ij - sum_{p < i} L_ip X_pj, one column per lane (lanes 0..15)
        const int b0 = 16 * w, jc = lane & 15;
        T y[16];
#pragma unroll
        for (int i = 0; i < 16; i++) {
            T s = i == jc ? T(1) : T(0);
#pragma unroll
            for (int p = 0; p < i; p++) s += s_l[b0 + i][b0 + p] * y[p];
            y[i] = s;
        }
        if (lane < 16)
#pragma unroll
            for (int i = 0; i < 16; i++) s_inv[w][i][jc] = y[i];
        __syncthreads();
    }
    const int ln = lane & 15, col = col0 + 16 * w + ln;
    const bool act = col < colend;
    T* ac = a + (int64_t)col * lda;
    typename M::vacc x[4];
    if (solve) {
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 16 * b + M::k(lane, r);
                x[b][r] = (act && row < kb) ? ac[s_map[row]] : T(0);
            }
    }
    // the interchanges (with U12: those into rows below the block), 32 pairs per lane group of 16
    T v[2 * NB / 4];
#pragma unroll
    for (int u = 0; u < 2 * NB / 4; u++) {
        const int e = 4 * u + (lane >> 4);
        if (4 * u < cnt) v[u] = (act && e < cnt) ? ac[s_ps[e]] : T(0);
    }
#pragma unroll
    for (int u = 0; u < 2 * NB / 4; u++) {
        const int e = 4 * u + (lane >> 4);
        if (4 * u < cnt && act && e < cnt) {
            const int d = s_pd[e];
            if (!solve || d < k0 || d >= k0 + kb) ac[d] = v[u];
        }
    }
    if (!solve) return;
#pragma unroll
    for (int b = 0; b < 4; b++) {
#pragma unroll
        for (int c = 0; c < b; c++)
#pragma unroll
            for (int r = 0; r < 4; r++) x[b] = M::mfma(s_l[16 * b + ln][16 * c + M::k(lane, r)], x[c][r], x[b]);
        typename M::vacc s = {T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int r = 0; r < 4; r++) s = M::mfma(s_inv[b][ln][M::k(lane, r)], x[b][r], s);
        // s += inv (x_b - L_bb s), the unit diagonal's part first
        x[b] -= s;
#pragma unroll
        for (int r = 0; r < 4; r++) x[b] = M::mfma(s_l[16 * b + ln][16 * b + M::k(lane, r)], s[r], x[b]);
#pragma unroll
        for (int r = 0; r < 4; r++) s = M::mfma(s_inv[b][ln][M::k(lane, r)], x[b][r], s);
        x[b] = s;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = 16 * b + M::k(lane, r);
            if (act && row < kb) ac[k0 + row] = x[b][r];
        }
    }
}

// C(m x n) -= A(m x kb) B(kb x n), the trailing update, on the matrix cores (any kb; batched over
// blockIdx.z with one stride for A, B and C).  One work-group of 4 waves per TI x TJ tile of C,
// waves arranged WAVES_I x (4 / WAVES_I) over it; each wave holds its block as NBI x NBJ MFMA
// blocks (FP32: v_mfma_f32_32x32x2f32, FP64: v_mfma_f64_16x16x4f64).  Operand layouts on gfx950:
// first operand lane l = P(l % BM, l / BM), second Q(l / BM, l % BM) (m, k and k, n); output
// register r of lane l = D(drow(l, r), l % BM).  The kernel computes D = (A B)^T block by block
// (P from B, Q from A), so that each lane's outputs lie along a column of C and the 64 lanes of one
// register read or write whole 128-byte row runs of C.
// A and B pass through LDS in 16-deep k-slices, double-buffered: the global loads of slice s + 1
// are in flight while the MFMAs consume slice s.  The accumulators start from zero and C is read
// once, in the epilogue (C - A B, the order of a BLAS gemm with alpha = -1, beta = 1).
// Tiles: FP32 128 x 64 (4 waves along the rows), 64 x 64 (2 x 2 waves) when the 128-row grid
// would hold fewer than 1024 work-groups; FP64 64 x 64 (4 waves along the rows).  Measured against
// rocBLAS ?gemm_strided_batched at k = 64: 2.79 vs 2.14 ms (m = n = 4032, batch 64, FP32),
// 0.73 vs 0.56 ms (m = n = 16320, FP32), 1.24 vs 1.04 ms (m = n = 16320, FP64).
template <typename T>
struct UpdCfg;
template <>
struct UpdCfg<float> {
    static constexpr int BM = 32, KS = 2, NACC = 16;
    typedef float vacc __attribute__((ext_vector_type(16)));
    static __device__ __forceinline__ vacc mfma(float p, float q, vacc c) {
        return __builtin_amdgcn_mfma_f32_32x32x2f32(p, q, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int drow(int l, int r) { return 8 * (r >> 2) + 4 * (l >> 5) + (r & 3); }
};
template <>
struct UpdCfg<double> {
    static constexpr int BM = 16, KS = 4, NACC = 4;
    typedef double vacc __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ vacc mfma(double p, double q, vacc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(p, q, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int drow(int l, int r) { return (l >> 4) + 4 * r; }
};

constexpr int kUpdDK = 16;  // k-slice depth
// Leading dimensions below this keep k_update's per-lane offsets (at most 15 of them and 15) in 32 bits, unsigned.
constexpr int64_t kUpdMaxLd = (int64_t)1 << 28;

// The FP32 128 x 64 tile is held to 6 waves per SIMD (its accumulators then sit in 80 vector registers
// beside the operands instead of 32 accumulation registers: 5 -> 6 waves; measured ~1 % on getrf).
template <typename T, int TI, int TJ, int WAVES_I>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 && TI * TJ == 8192 ? 6 : 1)))
void k_update(T* __restrict__ C, int64_t ldc, const T* __restrict__ A, int64_t lda, const T* __restrict__ B,
              int64_t ldb, int m, int n, int kb, int64_t sbatch) {
    using G = UpdCfg<T>;
    constexpr int BM = G::BM, KS = G::KS, DK = kUpdDK;
    constexpr int WI = TI / WAVES_I, WJ = TJ / (4 / WAVES_I), NBI = WI / BM, NBJ = WJ / BM;
    constexpr int NA = TI * DK / 256, NBq = TJ * DK / 256;  // staged elements per thread and slice
    static_assert(NBI >= 1 && NBJ >= 1 && NA >= 1 && NBq >= 1 && 256 % TI == 0, "tile shape");
    __shared__ T sa[2][DK][TI];
    __shared__ T sb[2][TJ][DK + 1];
    const int i0 = blockIdx.x * TI, j0 = blockIdx.y * TJ;
    // uniform tile bases: every per-lane offset below fits 32 bits (kUpdMaxLd)
    C += (int64_t)blockIdx.z * sbatch + i0 + (int64_t)j0 * ldc;
    A += (int64_t)blockIdx.z * sbatch + i0;
    B += (int64_t)blockIdx.z * sbatch + (int64_t)j0 * ldb;
    m -= i0;
    n -= j0;
    const int t = threadIdx.x, l = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wi = (w % WAVES_I) * WI, wj = (w / WAVES_I) * WJ;
    const int li = l % BM, lg = l / BM;
    const int ta_i = t % TI, ta_k = t / TI;  // A staging: rows along the threads
    const int tb_k = t % DK, tb_j = t / DK;  // B staging: k along the threads
    const unsigned offA = ta_i + ta_k * (unsigned)lda, offB = tb_k + tb_j * (unsigned)ldb;
    const int nsl = (kb + DK - 1) / DK;
    T ra[NA], rb[NBq];
    auto load = [&](int s) {
        const int k0 = s * DK;
        const T* Ak = A + (int64_t)k0 * lda;
#pragma unroll
        for (int q = 0; q < NA; q++) {
            const int k = k0 + ta_k + q * (256 / TI);
            ra[q] = (ta_i < m && k < kb) ? Ak[(int64_t)(q * (256 / TI)) * lda + offA] : T(0);
        }
        const T* Bk = B + k0;
#pragma unroll
        for (int q = 0; q < NBq; q++) {
            const int j = tb_j + q * (256 / DK);
            rb[q] = (j < n && k0 + tb_k < kb) ? Bk[(int64_t)(q * (256 / DK)) * ldb + offB] : T(0);
        }
    };
    load(0);
    typename G::vacc acc[NBI][NBJ];
#pragma unroll
    for (int bi = 0; bi < NBI; bi++)
#pragma unroll
        for (int bj = 0; bj < NBJ; bj++)
#pragma unroll
            for (int r = 0; r < G::NACC; r++) acc[bi][bj][r] = T(0);
    for (int s = 0; s < nsl; s++) {
        const int buf = s & 1;
        // buffer buf was last read in slice s - 2, which every wave finished before the barrier of s - 1
#pragma unroll
        for (int q = 0; q < NA; q++) sa[buf][ta_k + q * (256 / TI)][ta_i] = ra[q];
#pragma unroll
        for (int q = 0; q < NBq; q++) sb[buf][tb_j + q * (256 / DK)][tb_k] = rb[q];
        __syncthreads();
        if (s + 1 < nsl) load(s + 1);
#pragma unroll
        for (int kk = 0; kk < DK; kk += KS) {
            T a[NBI], b[NBJ];
#pragma unroll
            for (int bi = 0; bi < NBI; bi++) a[bi] = sa[buf][kk + lg][wi + bi * BM + li];
#pragma unroll
            for (int bj = 0; bj < NBJ; bj++) b[bj] = sb[buf][wj + bj * BM + li][kk + lg];
#pragma unroll
            for (int bi = 0; bi < NBI; bi++)
#pragma unroll
                for (int bj = 0; bj < NBJ; bj++) acc[bi][bj] = G::mfma(b[bj], a[bi], acc[bi][bj]);
        }
    }
    const unsigned offC = li + G::drow(l, 0) * (unsigned)ldc;
#pragma unroll
    for (int bi = 0; bi < NBI; bi++) {
        const int i = wi + bi * BM + li;
#pragma unroll
        for (int bj = 0; bj < NBJ; bj++) {
            T cv[G::NACC];
#pragma unroll
            for (int r = 0; r < G::NACC; r++) {
                const int j = wj + bj * BM + G::drow(l, r);
                const T* Cp = C + (wi + bi * BM) + (int64_t)(wj + bj * BM + G::drow(0, r)) * ldc;
                cv[r] = (i < m && j < n) ? __builtin_nontemporal_load(Cp + offC) : T(0);
            }
#pragma unroll
            for (int r = 0; r < G::NACC; r++) {
                const int j = wj + bj * BM + G::drow(l, r);
                T* Cp = C + (wi + bi * BM) + (int64_t)(wj + bj * BM + G::drow(0, r)) * ldc;
                if (i < m && j < n) __builtin_nontemporal_store(cv[r] - acc[bi][bj][r], Cp + offC);
            }
        }
    }
}

template <typename T>
void launch_update(T* C, int64_t ldc, const T* A, int64_t lda, const T* B, int64_t ldb, int m, int n, int kb,
                   int64_t sb, int batch, hipStream_t st) {
    if (m <= 0 || n <= 0 || kb <= 0) return;
    if constexpr (sizeof(T) == 4) {
        const int64_t tall = (int64_t)((m + 127) / 128) * ((n + 63) / 64) * batch;
        if (tall >= 1024)
            hipLaunchKernelGGL((k_update<T, 128, 64, 4>), dim3((m + 127) / 128, (n + 63) / 64, batch), dim3(256), 0, st,
                               C, ldc, A, lda, B, ldb, m, n, kb, sb);
        else
            hipLaunchKernelGGL((k_update<T, 64, 64, 2>), dim3((m + 63) / 64, (n + 63) / 64, batch), dim3(256), 0, st, C,
                               ldc, A, lda, B, ldb, m, n, kb, sb);
    } else {
        hipLaunchKernelGGL((k_update<T, 64, 64, 4>), dim3((m + 63) / 64, (n + 63) / 64, batch), dim3(256), 0, st, C, ldc,
                           A, lda, B, ldb, m, n, kb, sb);
    }
}

template <typename T, int NT, int Q, int IB>
int launch_panel_reg(T* a, int64_t lda, int n, int k0, int kb, int32_t* ipiv, int32_t* info, int32_t* perm,
                     hipStream_t st, int batch, int64_t sb, const SpecBufs<T>& sp) {
    // after a speculative panel, further work-groups that copy its last round's result where it stood
    const int copies = sp.on ? (n - k0 + NT - 1) / NT : 1;
    hipLaunchKernelGGL((k_panel_reg<T, NT, Q, IB>), dim3(copies, 1, batch), dim3(NT), 0, st, a, lda, n, k0, kb, ipiv,
                       info, perm, sb, sp);
    TVLM_LAUNCHED();
    return TVLM_OK;
}

// 256 threads (one wave per SIMD: no wave waits for issue slots, up to 512 registers per lane), rows
// per thread Q and sub-panel width IB per panel height, chosen so that the sub-panel (Q x IB values
// per thread) and its L-block buffers stay in registers.
template <typename T>
int panel_one_group(T* a, int64_t lda, int n, int k0, int kb, int32_t* ipiv, int32_t* info, int32_t* perm,
                    hipStream_t st, int batch, int64_t sb, const SpecBufs<T>& sp) {
    const int m = n - k0;
    if (m <= 256) return launch_panel_reg<T, 256, 1, 8>(a, lda, n, k0, kb, ipiv, info, perm, st, batch, sb, sp);
    if (m <= 512) return launch_panel_reg<T, 256, 2, 8>(a, lda, n, k0, kb, ipiv, info, perm, st, batch, sb, sp);
    if (m <= 1024) return launch_panel_reg<T, 256, 4, 8>(a, lda, n, k0, kb, ipiv, info, perm, st, batch, sb, sp);
    if (m <= 2048) return launch_panel_reg<T, 256, 8, 8>(a, lda, n, k0, kb, ipiv, info, perm, st, batch, sb, sp);
    if constexpr (sizeof(T) == 8) {
        if (m <= 4096) return launch_panel_reg<T, 256, 16, 4>(a, lda, n, k0, kb, ipiv, info, perm, st, batch, sb, sp);
        return launch_panel_reg<T, 256, 32, 2>(a, lda, n, k0, kb, ipiv, info, perm, st, batch, sb, sp);
    } else {
        if (m <= 4096) return launch_panel_reg<T, 256, 16, 4>(a, lda, n, k0, kb, ipiv, info, perm, st, batch, sb, sp);
        return launch_panel_reg<T, 256, 32, 4>(a, lda, n, k0, kb, ipiv, info, perm, st, batch, sb, sp);
    }
}

// Device buffers of a factorisation's speculative panels (one set of keys and flags per panel, cleared
// once): SpecWork::panel(kp) gives the panel's, the results' buffer is shared.
template <typename T>
struct SpecWork {
    SpecBufs<T> base;  // base.on = false: panels without speculation
    SpecBufs<T> panel(int kp) const {
        SpecBufs<T> b = base;
        const int64_t s = kp / NB, batch = base.batch;
        if (base.ldw - kp <= spec_min_rows<T>(batch)) b.on = false;
        if ((size_t)s < keyed(base.ldw))
            b.keys += s * (kSpecRounds - 1) * batch * kSpecSlots * NB;
        else
            b.keys = nullptr, b.rounds = 2;
        b.fail += s * kSpecRounds * batch;
        return b;
    }
    // panels with more rows below their first NB than round 2 has candidates
    static size_t keyed(int64_t n) { return n > 2 * NB ? (size_t)(n - 2 * NB + NB - 1) / NB : 0; }
    // bytes of the flags, the failure counts and the keys (zeroed before the first panel), and in all
    static size_t zeroed(int n, int batch) {
        const size_t panels = (size_t)(n + NB - 1) / NB;
        return (sizeof(unsigned long long) * keyed(n) * (kSpecRounds - 1) * kSpecSlots * NB +
                sizeof(int32_t) * (kSpecRounds * panels + 1)) * batch;
    }
    static size_t bytes(int n, int batch) {
        return (zeroed(n, batch) + 255) / 256 * 256 + sizeof(T) * (size_t)n * NB * batch;
    }
    void place(void* ws, int n, int batch) {
        base.batch = batch;
        const size_t panels = (size_t)(n + NB - 1) / NB;
        base.on = true;
        base.keys = static_cast<unsigned long long*>(ws);
        base.fail = reinterpret_cast<int32_t*>(base.keys + keyed(n) * (kSpecRounds - 1) * batch * kSpecSlots * NB);
        base.ostate = base.fail + kSpecRounds * panels * batch;
        base.w = reinterpret_cast<T*>(static_cast<char*>(ws) + (zeroed(n, batch) + 255) / 256 * 256);
        base.ldw = n;
    }
};

// The speculative rounds of the panel at kp; what they leave open (and the copy of the last round's
// result) is the caller's next launch: panel_one_group or panel_coop with the same buffers.
// Shares of the rows: 64 rows per work-group, but at most one work-group per CU in all: each factors the
// candidates again, and a second one on a CU has its chain on the same SIMD at the same time (32 FP32
// matrices of 4096 rows: rounds 2 and 3 took 189 us on average with two per CU).
template <typename T>
int panel_spec(T* a, int64_t lda, int n, int kp, int kb, int32_t* ipiv, int32_t* perm, hipStream_t st, int batch,
               int64_t sb, const SpecBufs<T>& sp) {
    int shares = (n - kp - kb + 63) / 64;
    const int most = batch < 128 ? 256 / batch - 1 : 1;
    if (shares > most) shares = most;
    const dim3 grid(shares + 1, 1, batch);  // one more for the candidates' result
    hipLaunchKernelGGL((k_panel_spec<T, 1>), grid, dim3(256), 0, st, a, lda, n, kp, kb, ipiv, perm, sb, sp, 1);
    TVLM_LAUNCHED();
    for (int round = 2; round <= sp.rounds; round++) {
        hipLaunchKernelGGL((k_panel_spec<T, 2>), grid, dim3(256), 0, st, a, lda, n, kp, kb, ipiv, perm, sb, sp, round);
        TVLM_LAUNCHED();
    }
    return TVLM_OK;
}

// One panel in one work-group per matrix, after the speculative rounds where the factorisation has them.
template <typename T>
int panel_fast(T* a, int64_t lda, int n, int kp, int kb, int32_t* ipiv, int32_t* info, int32_t* perm, hipStream_t st,
               int batch, int64_t sb, const SpecWork<T>& spec) {
    SpecBufs<T> sp;
    if (spec.base.on) sp = spec.panel(kp);
    if (sp.on) TVLM_TRY(panel_spec<T>(a, lda, n, kp, kb, ipiv, perm, st, batch, sb, sp));
    return panel_one_group<T>(a, lda, n, kp, kb, ipiv, info, perm, st, batch, sb, sp);
}

constexpr int kFastPanelRows = 8192;  // taller panels take the column-by-column panel
constexpr int kWidePanelBatch = 8;     // batches of at least this many matrices use 64-column panels

// ---- getrs ------------------------------------------------------------------------------------
template <typename T>
__global__ void k_apply_pivots(T* __restrict__ x, int64_t ldx, int n, const int32_t* __restrict__ ipiv) {
    T* xc = x + (int64_t)blockIdx.x * ldx;
    if (threadIdx.x != 0) return;
    for (int k = 0; k < n; k++) {
        const int p = ipiv[k] - 1;
        if (p != k) {
            const T tmp = xc[k];
            xc[k] = xc[p];
            xc[p] = tmp;
        }
    }
}

constexpr int SB = 256;  // diagonal block of the blocked solve

// Diagonal block solve: lower (unit) if LOWER, else upper; rows [r0, r0+nb); one WG per rhs.
template <typename T, bool LOWER>
__global__ __launch_bounds__(SB) void k_diag_solve(const T* __restrict__ a, int64_t lda, int r0, int nb,
                                                   T* __restrict__ x, int64_t ldx) {
    __shared__ T xs[SB];
    T* xc = x + (int64_t)blockIdx.x * ldx + r0;
    const int t = threadIdx.x;
    if (t < nb) xs[t] = xc[t];
    __syncthreads();
    if (LOWER) {
        for (int k = 0; k < nb; k++) {
            const T xk = xs[k];
            if (t > k && t < nb) xs[t] -= a[(r0 + t) + (int64_t)(r0 + k) * lda] * xk;
            __syncthreads();
        }
    } else {
        for (int k = nb - 1; k >= 0; k--) {
            if (t == 0) xs[k] = xs[k] / a[(r0 + k) + (int64_t)(r0 + k) * lda];
            __syncthreads();
            const T xk = xs[k];
            if (t < k) xs[t] -= a[(r0 + t) + (int64_t)(r0 + k) * lda] * xk;
            __syncthreads();
        }
    }
    if (t < nb) xc[t] = xs[t];
}

// x(rows [q0, q1)) -= A(rows [q0,q1), cols [c0, c0+nb)) x(c0 : c0+nb); one thread per row, per rhs.
template <typename T>
__global__ void k_off_update(const T* __restrict__ a, int64_t lda, int q0, int q1, int c0, int nb, T* __restrict__ x,
                             int64_t ldx) {
    __shared__ T xb[SB];
    T* xc = x + (int64_t)blockIdx.y * ldx;
    for (int e = threadIdx.x; e < nb; e += blockDim.x) xb[e] = xc[c0 + e];
    __syncthreads();
    const int i = q0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= q1) return;
    T s = T(0);
    for (int c = 0; c < nb; c++) s += a[i + (int64_t)(c0 + c) * lda] * xb[c];
    xc[i] -= s;
}

template <typename T>
__global__ void k_zero_info_batch(int32_t* info, int batch) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < batch) info[i] = 0;
}

// Work-groups for a cooperative panel of m rows, or 0 when the panel stays in one work-group (short
// panels, batches whose groups would not all fit in kCoopMaxGroups, or panels taller than the
// groups can hold).
template <typename T>
int coop_groups(int m, int batch) {
    if (m <= kCoopMinRows) return 0;
    const int per_group = coop_threads<T>();
    const int G = (m + per_group - 1) / per_group;
    if (G < 2 || G * batch > kCoopMaxGroups) return 0;
    return G;
}

__global__ void k_fill_i32(int32_t* __restrict__ p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

constexpr size_t kCoopLdsBytes = 128 * 1024;  // NT rows x NB columns (coop_threads)

std::atomic<unsigned> g_coop_spin_limit{kCoopSpinLimit};

// info[z] = kCoopStalled for every matrix a cooperative panel's wait gave up on (by any group)
__global__ void k_coop_fail_info(const int32_t* __restrict__ fail, int32_t* __restrict__ info, int batch) {
    const int z = blockIdx.x * blockDim.x + threadIdx.x;
    if (z < batch && fail[z] != 0) info[z] = kCoopStalled;
}

template <typename T>
int panel_coop(T* a, int64_t lda, int n, int k0, int kb, int G, int32_t* ipiv, int32_t* info, int32_t* perm,
               hipStream_t st, int batch, int64_t sb, int32_t* ctr, T* cval, int32_t* crow, T* xrow, int32_t* fail,
               const SpecBufs<T>& sp) {
    constexpr int NT = coop_threads<T>();
    static const hipError_t lds_attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_panel_coop<T, NT>),
                                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                                           (int)kCoopLdsBytes);
    TVLM_HIP(lds_attr);
    TVLM_REQUIRE(G >= 2 && G * batch <= kCoopMaxGroups && kb <= NB && (int64_t)G * NT >= (int64_t)(n - k0),
                 "cooperative panel: %d groups for %d rows", G, n - k0);
    TVLM_REQUIRE(ctr && cval && crow && xrow && fail, "cooperative panel without exchange buffers");
    hipLaunchKernelGGL((k_panel_coop<T, NT>), dim3(G, 1, batch), dim3(NT), kCoopLdsBytes, st, a, lda, n, k0, kb, G,
                       ipiv, info, perm, sb, ctr, cval, crow, xrow, g_coop_spin_limit.load(), fail, sp);
    TVLM_LAUNCHED();
    return TVLM_OK;
}

// shape[2] > 1 factors a batch of matrices, matrix b at ptr + b * stride[2]; ipiv holds n entries
// per matrix (matrix b at ipiv + b n), info one per matrix.
// Side stream and events of the batched look-ahead, one set per (device, caller stream), created
// on first use (default priority).  Per caller stream, so that factorisations running
// concurrently on different streams each have their own side chain.  The side stream is created
// with an all-CUs mask: such a stream gets a hardware queue of its own, so its updates can overlap
// the caller's panels whatever queue the caller's stream shares (streams without a mask share a
// small pool of queues, and two streams on one queue run one after the other).
struct LookaheadStreams {
    hipStream_t side = nullptr;
    hipEvent_t narrow_done = nullptr, rest_done = nullptr;
};

std::mutex g_lookahead_mu;
std::map<std::pair<int, hipStream_t>, LookaheadStreams> g_lookahead;

int lookahead_streams(hipStream_t caller, LookaheadStreams** out) {
    int dev = 0;
    TVLM_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(g_lookahead_mu);
    LookaheadStreams& L = g_lookahead[std::make_pair(dev, caller)];
    if (!L.side) {
        TVLM_TRY(create_queue_stream(&L.side));
        TVLM_HIP(hipEventCreateWithFlags(&L.narrow_done, hipEventDisableTiming));
        TVLM_HIP(hipEventCreateWithFlags(&L.rest_done, hipEventDisableTiming));
    }
    *out = &L;
    return TVLM_OK;
}

// Batched getrf with a one-panel look-ahead (batches of kWidePanelBatch or more, n <= kFastPanelRows,
// 64-column panels).  After panel k's interchanges and U12 (k_swap_trsm), the trailing update is
// split: the next panel's 64 columns are updated first on the caller's stream, which then factors
// panel k+1 at once, while the rest of the trailing update runs on a side stream; the next
// k_swap_trsm waits for both.  The panels (one work-group per matrix) thus run beside the
// bandwidth-bound updates instead of between them.  Same arithmetic as the plain loop.
// Batched look-ahead factorisation.  Each step starts from a factored block [k0, j1) (one or two
// panels) whose U12 is known on every column right of it, and the trailing matrix not yet updated by
// that block.  The caller's stream updates the step's own columns first and factors them at once,
// while the rest of the trailing update runs on a side stream; what touches the rest (interchanges,
// U12) waits for it.  While the batch's trailing matrices exceed the last-level cache
// (kLookaheadPairBytes) a step takes two panels A and B: A, A's interchanges and U12 on B's columns
// only, B's columns updated by A, B, B's interchanges on A's columns -- all inside the step's 128
// columns, beside the side stream -- then, after it, A's and B's interchanges on the columns left
// and right of the step (in that order), A's U12 on the right, B's rows right of the step updated by
// A, B's U12.  The next trailing update is then one of rank 2 NB: the trailing matrices are read and
// written once per two panels.  perm holds two panels' composed interchanges (A's, then B's).
constexpr double kLookaheadPairBytes = 256.0 * 1024 * 1024;

template <typename T>
int getrf_lookahead(T* a, int64_t lda, int n, int batch, int64_t sb, int32_t* ipiv, int32_t* info, int32_t* perm,
                    hipStream_t st, const SpecWork<T>& spec) {
    LookaheadStreams* L = nullptr;
    TVLM_TRY(lookahead_streams(st, &L));
    int32_t* perm2 = perm + (size_t)batch * kPermInts;
    // interchanges (mode 0/1) and U12 (mode 0/2) of the panel at kp on nleft blocks of 64 columns
    // from lbase and nright blocks from rbase
    auto swaps = [&](int kp, int kb, const int32_t* pm, int mode, int lbase, int nleft, int rbase, int nright) -> int {
        if (nleft + nright > 0) {
            hipLaunchKernelGGL(k_swap_trsm<T>, dim3(nleft + nright, 1, batch), dim3(256), 0, st, a, lda, n, kp, kb,
                               nleft, pm, sb, mode, 0, nullptr, lbase, rbase);
            TVLM_LAUNCHED();
        }
        return TVLM_OK;
    };
    auto blocks = [](int cols) { return cols > 0 ? (cols + 63) / 64 : 0; };
    auto at = [&](int r, int c) { return a + r + (int64_t)c * lda; };
    int k0 = 0, j1 = n < NB ? n : NB;
    TVLM_TRY(panel_fast<T>(a, lda, n, k0, j1, ipiv, info, perm, st, batch, sb, spec));
    TVLM_TRY(swaps(k0, j1, perm, 0, 0, 0, j1, blocks(n - j1)));
    while (j1 < n) {
        const int kr = j1 - k0, m = n - j1;  // rank of the pending update; trailing size
        const double tail = (double)batch * (double)m * (double)m * sizeof(T);
        const bool pair = m > 2 * NB && tail > kLookaheadPairBytes;
        const int w = pair ? 2 * NB : (m < NB ? m : NB), jw = j1 + w;  // the step's columns [j1, jw)
        launch_update<T>(at(j1, j1), lda, at(j1, k0), lda, at(k0, j1), lda, m, w, kr, sb, batch, st);
        TVLM_LAUNCHED();
        const bool rest = m > w;
        if (rest) {
            TVLM_HIP(hipEventRecord(L->narrow_done, st));
            TVLM_HIP(hipStreamWaitEvent(L->side, L->narrow_done, 0));
            launch_update<T>(at(j1, jw), lda, at(j1, k0), lda, at(k0, jw), lda, m, m - w, kr, sb, batch, L->side);
            TVLM_LAUNCHED();
            TVLM_HIP(hipEventRecord(L->rest_done, L->side));
        }
        if (!pair) {
            TVLM_TRY(panel_fast<T>(a, lda, n, j1, w, ipiv, info, perm, st, batch, sb, spec));
            if (rest) TVLM_HIP(hipStreamWaitEvent(st, L->rest_done, 0));
            TVLM_TRY(swaps(j1, w, perm, 0, 0, blocks(j1), jw, blocks(n - jw)));
            k0 = j1;
            j1 = jw;
            continue;
        }
        const int jA = j1 + NB;  // panel A = [j1, jA), panel B = [jA, jw)
        TVLM_TRY(panel_fast<T>(a, lda, n, j1, NB, ipiv, info, perm, st, batch, sb, spec));
        TVLM_TRY(swaps(j1, NB, perm, 0, 0, 0, jA, 1));
        launch_update<T>(at(jA, jA), lda, at(jA, j1), lda, at(j1, jA), lda, n - jA, NB, NB, sb, batch, st);
        TVLM_LAUNCHED();
        TVLM_TRY(panel_fast<T>(a, lda, n, jA, NB, ipiv, info, perm2, st, batch, sb, spec));
        TVLM_TRY(swaps(jA, NB, perm2, 1, j1, 1, 0, 0));
        if (rest) TVLM_HIP(hipStreamWaitEvent(st, L->rest_done, 0));
        TVLM_TRY(swaps(j1, NB, perm, 1, 0, blocks(j1), jw, blocks(n - jw)));
        TVLM_TRY(swaps(jA, NB, perm2, 1, 0, blocks(j1), jw, blocks(n - jw)));
        if (jw < n) {
            TVLM_TRY(swaps(j1, NB, perm, 2, 0, 0, jw, blocks(n - jw)));
            launch_update<T>(at(jA, jw), lda, at(jA, j1), lda, at(j1, jw), lda, NB, n - jw, NB, sb, batch, st);
            TVLM_LAUNCHED();
            TVLM_TRY(swaps(jA, NB, perm2, 2, 0, 0, jw, blocks(n - jw)));
        }
        k0 = j1;
        j1 = jw;
    }
    return TVLM_OK;
}

// ---- deferred interchanges of the L columns (cooperative factorisations) ------------------------
//
// LAPACK's getrf applies every panel's row interchanges to all columns left of the panel.  The
// cooperative factorisation applies them only to the columns that a later step still reads (the
// first panel of a pair takes the second's).  Every other column block P (columns [NB P, NB P + NB))
// keeps a gather list g_P of n rows instead, identity at the start: each later panel's composed
// interchanges (dst <- src pairs) update the list, g[dst] = g[src] (a few hundred integers, in
// k_swap_trsm), instead of two scattered rows per pair in each of the block's columns.  At the end
// k_defer_gather (one work-group per column) stages rows [NB (P + 1), n) of its column in LDS and
// writes row r back from row g_P[r]: one contiguous pass over L.  The lists only move rows at or
// below NB (P + 1), so g_P[r] stays in [NB (P + 1), n) there.
constexpr size_t kDeferLdsBytes = 128 * 1024;  // rows [NB (P + 1), n) of one column

__global__ void k_iota_lists(int32_t* __restrict__ g, int n, int64_t total) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < total) g[i] = (int32_t)(i % n);
}

template <typename T>
__global__ __launch_bounds__(1024) void k_defer_gather(T* __restrict__ a, int64_t lda, int n,
                                                       const int32_t* __restrict__ gtab, int nblocks, int64_t sb) {
    extern __shared__ unsigned char s_raw[];
    T* s_col = reinterpret_cast<T*>(s_raw);
    const int c = blockIdx.x, P = c / NB, t = threadIdx.x;
    const int from = NB * (P + 1);
    if (from >= n) return;
    a += (int64_t)blockIdx.z * sb + (int64_t)c * lda;
    gtab += ((int64_t)blockIdx.z * nblocks + P) * n;
    const int m = n - from;
#pragma unroll 4
    for (int r = t; r < m; r += 1024) s_col[r] = a[from + r];
    __syncthreads();
#pragma unroll 4
    for (int r = t; r < m; r += 1024) {
        const int src = gtab[from + r] - from;
        a[from + r] = s_col[(unsigned)src < (unsigned)m ? src : r];
    }
}

template <typename T>
int defer_gather(T* a, int64_t lda, int n, int batch, int64_t sb, const int32_t* gtab, hipStream_t st) {
    const int nblocks = (n + NB - 1) / NB;
    if (nblocks < 2) return TVLM_OK;
    TVLM_REQUIRE((size_t)n * sizeof(T) <= kDeferLdsBytes, "deferred interchanges: n = %d too large", n);
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_defer_gather<T>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                                       (int)kDeferLdsBytes);
    TVLM_HIP(attr);
    hipLaunchKernelGGL(k_defer_gather<T>, dim3(n, 1, batch), dim3(1024), sizeof(T) * (size_t)n, st, a, lda, n, gtab,
                       nblocks, sb);
    TVLM_LAUNCHED();
    return TVLM_OK;
}

// Factorisations whose tall panels are cooperative (all panels NB wide), taken kGroupPanels panels at a
// time so that the trailing matrix is read and written once per group.  For each panel of a group: its
// columns updated by the group's earlier panels, the panel, its interchanges on both sides (mode 1; the
// group's first: and U12, mode 0), its rows right of it updated by the group's earlier panels, its U12
// (mode 2); then one update of the trailing matrix by the whole group.  The same products as one panel
// at a time, summed in a different order.
constexpr int kGroupPanels = 4;
constexpr int kGroupMinRows = 3072;  // trailing matrices at least this tall are updated once per group

// ---- the factorisation plan -------------------------------------------------------------------
// Which path a getrf call takes and, for the cooperative path, every panel's form and exchange
// buffers; computed on the host before anything is queued (getrf_plan), executed by getrf, and
// exported as tvlm_getrf_plan so that the schedule and the buffer sizing can be checked without a GPU.
//   kPathLookahead : batches of >= kWidePanelBatch matrices of <= kFastPanelRows rows (one-group panels
//                    beside the trailing updates on a side stream);
//   kPathCoop      : the first panel is cooperative; then every panel of more than kCoopMinRows rows is
//                    (coop_groups falls with the rows) and takes its own counter set;
//   kPathPanels    : one work-group per panel throughout (k_panel_reg, or the column-by-column k_panel
//                    above kFastPanelRows rows) -- also every factorisation with cooperative panels
//                    switched off.
enum GetrfPath { kPathLookahead = 0, kPathCoop = 1, kPathPanels = 2 };

struct GetrfStep {
    int kp, kb;   // first column and width of the panel
    int groups;   // work-groups of a cooperative panel, 0 for a one-group panel
    int ctr_set;  // counter set of a cooperative panel, -1 otherwise
};

struct GetrfPlan {
    int path = kPathPanels;
    std::vector<GetrfStep> steps;  // kPathCoop only
    int ctr_sets = 0;              // counter sets allocated (one per cooperative panel)
    // exchange buffers (kPathCoop): ints (counters, per-matrix failure word, candidate
    // rows, gather lists) and reals (candidate values, published rows)
    size_t nctr = 0, ncand = 0, nrow = 0, ngat = 0;
    size_t coop_bytes(size_t real_bytes) const {
        return nctr || ncand ? sizeof(int32_t) * (nctr + ncand + ngat) + real_bytes * (ncand + nrow) + 512 : 0;
    }
};

template <typename T>
GetrfPlan getrf_plan(int n, int batch, bool allow_coop) {
    GetrfPlan P;
    if (batch >= kWidePanelBatch && n <= kFastPanelRows) {
        P.path = kPathLookahead;
        return P;
    }
    if (!allow_coop || coop_groups<T>(n, batch) == 0) {
        P.path = kPathPanels;
        return P;
    }
    P.path = kPathCoop;
    for (int kp = 0; kp < n; kp += NB) {
        GetrfStep st{kp, n - kp < NB ? n - kp : NB, coop_groups<T>(n - kp, batch), -1};
        if (st.groups > 0) st.ctr_set = P.ctr_sets++;
        P.steps.push_back(st);
    }
    const int panels = (n + NB - 1) / NB;
    P.nctr = (size_t)P.ctr_sets * batch * kCoopCtr + 2 * (size_t)batch;  // (batch words would do)
    P.ncand = (size_t)batch * NB * kCoopMaxGroups;
    P.nrow = (size_t)batch * kCoopXrow;
    P.ngat = (size_t)batch * panels * n;
    return P;
}

template <typename T>
int getrf_coop(T* a, int64_t lda, int n, int batch, int64_t sb, int32_t* ipiv, int32_t* info, int32_t* perm,
                     hipStream_t st, const GetrfPlan& plan, int32_t* ctr, T* cval, int32_t* crow, T* xrow,
                     int32_t* gtab, int32_t* fail, const SpecWork<T>& spec) {
    if (n > NB) {
        const int64_t total = (int64_t)batch * ((n + NB - 1) / NB) * n;
        hipLaunchKernelGGL(k_iota_lists, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, gtab, n, total);
        TVLM_LAUNCHED();
    }
    auto panel = [&](int kp, int kb) -> int {
        // the planned panel at kp: its width, group count and exchange counter set
        const int s = kp / NB;
        TVLM_REQUIRE(kp % NB == 0 && s < (int)plan.steps.size() && plan.steps[s].kp == kp && plan.steps[s].kb == kb,
                     "panel at column %d (width %d) is not in the factorisation plan", kp, kb);
        const GetrfStep& p = plan.steps[s];
        if (p.groups == 0) return panel_fast<T>(a, lda, n, kp, kb, ipiv, info, perm, st, batch, sb, spec);
        TVLM_REQUIRE(p.ctr_set >= 0 && p.ctr_set < plan.ctr_sets, "cooperative panel %d: counter set %d of %d", s,
                     p.ctr_set, plan.ctr_sets);
        SpecBufs<T> sp;
        if (spec.base.on) sp = spec.panel(kp);
        if (sp.on) TVLM_TRY(panel_spec<T>(a, lda, n, kp, kb, ipiv, perm, st, batch, sb, sp));
        return panel_coop<T>(a, lda, n, kp, kb, p.groups, ipiv, info, perm, st, batch, sb,
                             ctr + (size_t)p.ctr_set * batch * kCoopCtr, cval, crow, xrow, fail, sp);
    };
    // the left columns before left0 take the interchanges into their gather lists
    auto swap_trsm = [&](int kp, int kb, int mode, int left0) -> int {
        const int j1 = kp + kb;
        const int nleft = mode == 2 ? 0 : (kp + 63) / 64, nright = (n - j1 + 63) / 64;
        if (nleft + nright > 0) {
            hipLaunchKernelGGL(k_swap_trsm<T>, dim3(nleft + nright, 1, batch), dim3(256), 0, st, a, lda, n, kp, kb,
                               nleft, perm, sb, mode, left0, gtab);
            TVLM_LAUNCHED();
        }
        return TVLM_OK;
    };
    auto at = [&](int r, int c) { return a + r + (int64_t)c * lda; };
    for (int kp = 0; kp < n;) {
        // a trailing matrix below kGroupMinRows stays in the last-level cache: one panel at a time
        const int last = kp + NB < n && n - kp - NB >= kGroupMinRows ? kp + kGroupPanels * NB : kp + NB;
        int c = kp;
        while (c < last && c < n) {
            const int kb = n - c < NB ? n - c : NB, j1 = c + kb, r = c - kp;  // r: rank of the group's panels so far
            if (r) {
                launch_update<T>(at(c, c), lda, at(c, kp), lda, at(kp, c), lda, n - c, kb, r, sb, batch, st);
                TVLM_LAUNCHED();
            }
            TVLM_TRY(panel(c, kb));
            TVLM_TRY(swap_trsm(c, kb, r ? 1 : 0, kp));
            if (r && j1 < n) {
                launch_update<T>(at(c, j1), lda, at(c, kp), lda, at(kp, j1), lda, kb, n - j1, r, sb, batch, st);
                TVLM_LAUNCHED();
                TVLM_TRY(swap_trsm(c, kb, 2, c));
            }
            c = j1;
        }
        if (c < n) {
            launch_update<T>(at(c, c), lda, at(c, kp), lda, at(kp, c), lda, n - c, n - c, c - kp, sb, batch, st);
            TVLM_LAUNCHED();
        }
        kp = c;
    }
    TVLM_TRY(defer_gather<T>(a, lda, n, batch, sb, gtab, st));
    hipLaunchKernelGGL(k_coop_fail_info, dim3((batch + 255) / 256), dim3(256), 0, st, fail, info, batch);
    TVLM_LAUNCHED();
    return TVLM_OK;
}

template <typename T>
int getrf(const tvlm_view* av, int32_t* ipiv, int32_t* info, void* stream, bool allow_coop = true) {
    TVLM_REQUIRE(av && av->ptr && ipiv && info, "null argument");
    TVLM_REQUIRE(av->stride[0] == 1, "A must be column-major");
    TVLM_REQUIRE(av->shape[0] == av->shape[1], "A must be square (got %lld x %lld)", (long long)av->shape[0],
                 (long long)av->shape[1]);
    const int n = (int)av->shape[0];
    const int batch = (int)av->shape[2];
    const int64_t lda = av->stride[1], sb = av->stride[2];
    TVLM_REQUIRE(lda >= n || n == 0, "lda < n");
    TVLM_REQUIRE(n <= NB || lda < kUpdMaxLd, "lda %lld out of range for a trailing update", (long long)lda);
    TVLM_REQUIRE(batch >= 1 && batch <= 65535, "batch %d out of range", batch);
    TVLM_REQUIRE(batch == 1 || sb >= lda * n, "matrices of the batch overlap (stride[2] < stride[1] * n)");
    hipStream_t st = as_stream(stream);
    T* a = static_cast<T*>(av->ptr);
    hipLaunchKernelGGL(k_zero_info_batch<T>, dim3((batch + 255) / 256), dim3(256), 0, st, info, batch);
    TVLM_LAUNCHED();
    void* ws = nullptr;
    TVLM_TRY(device_workspace(sizeof(int32_t) * kPermInts * 2 * (size_t)batch, &ws, kWsLuPerm, st));
    int32_t* perm = static_cast<int32_t*>(ws);
    const GetrfPlan plan = getrf_plan<T>(n, batch, allow_coop);
    void* cws = nullptr;
    if (plan.path == kPathCoop) TVLM_TRY(device_workspace(plan.coop_bytes(sizeof(T)), &cws, kWsLuCoop, st));
    // Speculative panels wherever a panel kernel of at most kFastPanelRows rows or a cooperative one
    // follows them.  With a spin limit set (a diagnostic), cooperative factorisations go without, so that
    // the waits it bounds are run.
    SpecWork<T> spec;
    // Without room for their buffers the panels go without as well.
    void* sws = nullptr;
    if (n > spec_min_rows<T>(batch) && n <= kSpecMaxRows &&
        (plan.path == kPathCoop ? g_coop_spin_limit.load() == kCoopSpinLimit : n <= kFastPanelRows)) {
        const int rc = device_workspace(SpecWork<T>::bytes(n, batch), &sws, kWsLuSpec, st);
        if (rc == TVLM_ERR_NOMEM)
            (void)hipGetLastError();
        else
            TVLM_TRY(rc);
    }
    if (sws) {
        spec.place(sws, n, batch);
        const int64_t words = (int64_t)(SpecWork<T>::zeroed(n, batch) / sizeof(int32_t));
        hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st,
                           static_cast<int32_t*>(sws), words);
        TVLM_LAUNCHED();
    }
    if (plan.path == kPathLookahead) return getrf_lookahead<T>(a, lda, n, batch, sb, ipiv, info, perm, st, spec);
    if (plan.path == kPathCoop) {
        // Buffers (sized by the plan): per cooperative panel and matrix kCoopCtr counters, per matrix
        // the failure word (all zeroed here, once for the whole factorisation), the candidates, the
        // published rows, and the deferred interchanges' gather lists.
        int32_t* ctr = static_cast<int32_t*>(cws);
        int32_t* crow = ctr + plan.nctr;
        T* cval = reinterpret_cast<T*>((reinterpret_cast<uintptr_t>(crow + plan.ncand) + 255) & ~(uintptr_t)255);
        T* xrow = cval + plan.ncand;
        int32_t* gtab =
            reinterpret_cast<int32_t*>((reinterpret_cast<uintptr_t>(xrow + plan.nrow) + 255) & ~(uintptr_t)255);
        hipLaunchKernelGGL(k_fill_i32, dim3((unsigned)((plan.nctr + 255) / 256)), dim3(256), 0, st, ctr,
                           (int64_t)plan.nctr);
        TVLM_LAUNCHED();
        int32_t* fail = ctr + (size_t)plan.ctr_sets * batch * kCoopCtr;  // per matrix: a wait gave up
        return getrf_coop<T>(a, lda, n, batch, sb, ipiv, info, perm, st, plan, ctr, cval, crow, xrow, gtab,
                                   fail, spec);
    }
    for (int k0 = 0; k0 < n;) {
        // tall panels of one matrix are narrower: the in-panel left-looking traffic grows with width
        // squared.  A batch is bound by the trailing updates instead, whose traffic (the whole
        // trailing matrix read and written per panel) halves with the full width.
        const int width = (!spec.base.on && n - k0 > 2048 && batch < kWidePanelBatch) ? NB / 2 : NB;
        const int kb = (n - k0 < width) ? n - k0 : width;
        const int j1 = k0 + kb;
        const int kp = k0;  // this panel's first column
        k0 = j1;
        if (n - kp <= kFastPanelRows) {
            TVLM_TRY(panel_fast<T>(a, lda, n, kp, kb, ipiv, info, perm, st, batch, sb, spec));
            const int nleft = (kp + 63) / 64, nright = (n - j1 + 63) / 64;
            if (nleft + nright > 0) {
                hipLaunchKernelGGL(k_swap_trsm<T>, dim3(nleft + nright, 1, batch), dim3(256), 0, st, a, lda, n, kp, kb,
                                   nleft, perm, sb);
                TVLM_LAUNCHED();
            }
        } else {
            for (int z = 0; z < batch; z++) {
                T* az = a + (int64_t)z * sb;
                int32_t* pz = ipiv + (int64_t)z * n;
                hipLaunchKernelGGL(k_panel<T>, dim3(1), dim3(kPanelThreads), 0, st, az, lda, n, kp, kb, pz, info + z);
                TVLM_LAUNCHED();
                if (kp > 0) {
                    hipLaunchKernelGGL(k_laswp<T>, dim3((kp + 255) / 256), dim3(256), 0, st, az, lda, 0, kp, kp, kb, pz);
                    TVLM_LAUNCHED();
                }
                if (j1 < n) {
                    hipLaunchKernelGGL(k_laswp<T>, dim3((n - j1 + 255) / 256), dim3(256), 0, st, az, lda, j1, n, kp, kb,
                                       pz);
                    TVLM_LAUNCHED();
                    hipLaunchKernelGGL(k_trsm<T>, dim3((n - j1 + 255) / 256), dim3(256), 0, st, az, lda, n, kp, kb, j1);
                    TVLM_LAUNCHED();
                }
            }
        }
        if (j1 >= n) continue;
        const int m = n - j1;
        launch_update<T>(a + j1 + (int64_t)j1 * lda, lda, a + j1 + (int64_t)kp * lda, lda, a + kp + (int64_t)j1 * lda,
                         lda, m, m, kb, sb, batch, st);
        TVLM_LAUNCHED();
    }
    return TVLM_OK;
}

// ---- blocked getrs ----------------------------------------------------------------------------
constexpr int kSB = 64;            // solve block
constexpr int kSW = 4 * kSB;       // rows of a substitution step
constexpr int kSolveMaxN = 16384;  // rhs column in LDS
constexpr int kSolvePairs = 1 + 2 * 2 * kSB;
constexpr int kBlockedMaxN = 1024;  // rhs column of k_solve_blocked in LDS (two work-groups a CU; with 16384 rows
                                    // one, and 1.3 times the time)

// y = 0: composes the interchanges of pivot block b (64 positions) into (dst, src) pairs (one wave);
// y = 1 / 2: inverts the 64 x 64 diagonal block b of L (unit lower) / U (upper): each wave one 16 x 16
// diagonal tile by substitution, a column per lane; then tile pairs and the two 32-row halves are merged by
// [A 0; B C]^-1 = [A^-1 0; -C^-1 B A^-1, C^-1] (U: its mirror image) on the matrix cores.  Bound by the chain of
// dependent steps: row by row over all 64 with the sums split over the waves it took 46 us, 32 times 8 blocks;
// 14 us so.
template <typename T>
__global__ __launch_bounds__(256) void k_solve_prep(const T* __restrict__ a, int64_t lda, int n,
                                                    const int32_t* __restrict__ ipiv, int32_t* __restrict__ pairs,
                                                    T* __restrict__ inv, int64_t sa) {
    using M = Mf16<T>;
    __shared__ int s_p[kSB];
    __shared__ int s_pd[2 * kSB], s_ps[2 * kSB];
    __shared__ T s_a[kSB][kSB + 1];
    __shared__ T s_x[kSB][kSB + 1];  // the inverse, row by row
    const int nb_ = (n + kSB - 1) / kSB;  // batch: one matrix per blockIdx.z
    a += (int64_t)blockIdx.z * sa;
    ipiv += (int64_t)blockIdx.z * n;
    pairs += (int64_t)blockIdx.z * nb_ * kSolvePairs;
    inv += (int64_t)blockIdx.z * 2 * nb_ * kSB * kSB;
    const int b = blockIdx.x, t = threadIdx.x, lane = t & 63, g = t >> 6;
    const int r0 = b * kSB, rb = min(kSB, n - r0);
    if (blockIdx.y == 0) {
        if (t < kSB && lane < rb) s_p[lane] = ipiv[r0 + lane] - 1;
        __syncthreads();
        if (t < kSB) {
            const int np = wave_compose_swaps(r0, rb, s_p, s_pd, s_ps);
            int32_t* out = pairs + (int64_t)b * kSolvePairs;
            for (int e = lane; e < np; e += 64) {
                out[1 + 2 * e] = s_pd[e];
                out[2 + 2 * e] = s_ps[e];
            }
            if (lane == 0) out[0] = np;
        }
        return;
    }
    const bool lower = blockIdx.y == 1;
    for (int e = t; e < kSB * kSB; e += 256) {
        const int r = e % kSB, c = e / kSB;
        s_a[r][c] = (r < rb && c < rb) ? a[(r0 + r) + (int64_t)(r0 + c) * lda] : (r == c ? T(1) : T(0));
        s_x[r][c] = T(0);
    }
    __syncthreads();
    const int m = lane & 15;
    {
        T v[16];
        const int o = 16 * g;
        if (lower) {
#pragma unroll
            for (int i = 0; i < 16; i++) {
                T sum = T(0);
#pragma unroll
                for (int p = 0; p < i; p++) sum += s_a[o + i][o + p] * v[p];
                v[i] = i < m ? T(0) : (i == m ? T(1) : -sum);
            }
        } else {
#pragma unroll
            for (int i = 15; i >= 0; i--) {
                T sum = T(0);
#pragma unroll
                for (int p = i + 1; p < 16; p++) sum += s_a[o + i][o + p] * v[p];
                v[i] = i > m ? T(0) : ((i == m ? T(1) : T(0)) - sum) / s_a[o + i][o + i];
            }
        }
        if (lane < 16)
#pragma unroll
            for (int i = 0; i < 16; i++) s_x[o + i][o + m] = v[i];
    }
    __syncthreads();
    typedef typename M::vacc vacc;
    // c + P(tile pi, pk of s) Q, Q a 16 x 16 tile in the second operand's layout
    auto mul = [&](const T(*P)[kSB + 1], int pi, int pk, const vacc& q, vacc c) {
#pragma unroll
        for (int r = 0; r < 4; r++) c = M::mfma(P[16 * pi + m][16 * pk + M::k(lane, r)], q[r], c);
        return c;
    };
    auto tile = [&](int ki, int kj) {
        vacc q;
#pragma unroll
        for (int r = 0; r < 4; r++) q[r] = s_x[16 * ki + M::k(lane, r)][16 * kj + m];
        return q;
    };
    auto put = [&](int ki, int kj, const vacc& q) {
#pragma unroll
        for (int r = 0; r < 4; r++) s_x[16 * ki + M::k(lane, r)][16 * kj + m] = -q[r];
    };
    const vacc zero = {T(0), T(0), T(0), T(0)};
    if (g < 2) {  // i: the tile row to form, k: the tile row it draws on
        const int i = lower ? 2 * g + 1 : 2 * g, k = lower ? 2 * g : 2 * g + 1;
        put(i, k, mul(s_x, i, i, mul(s_a, i, k, tile(k, k), zero), zero));
    }
    __syncthreads();
    {
        const int i0 = lower ? 2 : 0, q0 = lower ? 0 : 2;  // first tile row to form, first it draws on
        const int i = i0 + (g >> 1), col = q0 + (g & 1);
        const vacc x0 = tile(q0, col), x1 = tile(q0 + 1, col);
        const vacc t0 = mul(s_a, i0, q0 + 1, x1, mul(s_a, i0, q0, x0, zero));
        const vacc t1 = mul(s_a, i0 + 1, q0 + 1, x1, mul(s_a, i0 + 1, q0, x0, zero));
        vacc y = zero;
        if (lower ? true : i == i0) y = mul(s_x, i, i0, t0, y);
        if (lower ? i > i0 : true) y = mul(s_x, i, i0 + 1, t1, y);
        put(i, col, y);
    }
    __syncthreads();
    T* out = inv + ((int64_t)(lower ? 0 : 1) * ((n + kSB - 1) / kSB) + b) * kSB * kSB;
    for (int e = t; e < kSB * kSB; e += 256) {
        const int r = e % kSB, c = e / kSB;
        out[r + (int64_t)c * kSB] = s_x[r][c];
    }
}

// perm[i]: the row of the right-hand side that all interchanges bring to row i (one work-group per matrix;
// a block's list is in flight while the one before it is applied).  Pivots that a panel which gave up waiting
// never wrote are skipped: perm stays within the matrix.
__global__ __launch_bounds__(256) void k_solve_compose(int n, const int32_t* __restrict__ pairs,
                                                       int32_t* __restrict__ perm) {
    __shared__ int32_t s_i[kSolveMaxN];
    const int t = threadIdx.x;
    const int nblk = (n + kSB - 1) / kSB;
    pairs += (int64_t)blockIdx.x * nblk * kSolvePairs;
    perm += (int64_t)blockIdx.x * n;
    for (int i = t; i < n; i += 256) s_i[i] = i;
    auto load = [&](int b, int& np, int& dst, int& src) {  // at most 2 kSB = 128 pairs, all initialised ones read
        const int32_t* pl = pairs + (int64_t)b * kSolvePairs;
        np = pl[0];
        const int e = t < 2 * kSB ? t : 0;
        dst = pl[1 + 2 * e];
        src = pl[2 + 2 * e];
    };
    int np, dst, src;
    load(0, np, dst, src);
    __syncthreads();
    for (int b = 0; b < nblk; b++) {
        int np1 = 0, dst1 = 0, src1 = 0;
        if (b + 1 < nblk) load(b + 1, np1, dst1, src1);
        int v = 0;
        const bool mine = t < np && (unsigned)src < (unsigned)n && (unsigned)dst < (unsigned)n;
        if (mine) v = s_i[src];
        __syncthreads();
        if (mine) s_i[dst] = v;
        __syncthreads();
        np = np1, dst = dst1, src = src1;
    }
    for (int i = t; i < n; i += 256) perm[i] = s_i[i];
}

// The triangular tiles of kSW rows that finish them: thread (r, g) = (t & 63, t >> 6) holds columns 4 g .. 4 g + 3
// of row r, of the four diagonal blocks' inverses and of the off-diagonal tiles between them.
template <typename T, bool LOWER>
struct SolveTiles {
    T iv[4][4], off[6][4];
    static __device__ __forceinline__ constexpr int at(int q, int s) {  // index of tile (q, s), s before q
        return LOWER ? q * (q - 1) / 2 + s : (3 - q) * (2 - q) / 2 + (3 - s);
    }
    // a: the matrix at the step's first row and column, nr rows left from there (past them the last row or
    // column, or the first inverse, is read, and not used); inv: its blocks' inverses
    __device__ __forceinline__ void load(const T* __restrict__ a, int64_t lda, int nr, const T* __restrict__ inv, int r,
                                         int g) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
#pragma unroll
            for (int p = 0; p < 4; p++)
                iv[q][p] = (inv + (q * kSB < nr ? q : 0) * kSB * kSB + (4 * g + p) * kSB)[(unsigned)r];
#pragma unroll
            for (int s = 0; s < 4; s++)
                if (LOWER ? s < q : s > q) {
                    const unsigned row = min(q * kSB + r, nr - 1);
#pragma unroll
                    for (int p = 0; p < 4; p++) off[at(q, s)][p] = (a + (int64_t)min(s * kSB + 4 * g + p, nr - 1) * lda)[row];
                }
        }
    }
    // Substitution in the step's rows: x = its right-hand side (LDS), replaced by the solution; acc[q]: what
    // this thread's columns subtract from row q kSB + r already.  Rows past nr hold 0 and stay so.
    __device__ __forceinline__ void solve(T* x, T (*red)[kSB], T* yb, T acc[4], int nr, int t) const {
        const int r = t & 63, g = __builtin_amdgcn_readfirstlane(t >> 6);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int q = LOWER ? e : 3 - e;
            if (q * kSB >= nr) continue;  // uniform over the work-group
            red[g][r] = acc[q];
            __syncthreads();
            if (t < kSB) {
                T y = x[q * kSB + t];
#pragma unroll
                for (int k = 0; k < 16; k++) y -= red[k][t];
                yb[t] = q * kSB + t < nr ? y : T(0);
            }
            __syncthreads();
            T s = T(0);
#pragma unroll
            for (int p = 0; p < 4; p++) s += iv[q][p] * yb[4 * g + p];
            red[g][r] = s;
            __syncthreads();
            if (t < kSB) {
                T v = T(0);
#pragma unroll
                for (int k = 0; k < 16; k++) v += red[k][t];
                x[q * kSB + t] = q * kSB + t < nr ? v : T(0);
            }
            __syncthreads();
#pragma unroll
            for (int w = 0; w < 4; w++)
                if (LOWER ? w > q : w < q)
#pragma unroll
                    for (int p = 0; p < 4; p++)
                        if (q * kSB + 4 * g + p < nr) acc[w] += off[at(w, q)][p] * x[q * kSB + 4 * g + p];
        }
    }
};

// n <= kSW: one work-group per right-hand side, its column in LDS.
// The whole chain is latency (8 dependent 64-row steps): the tiles are in registers before it starts.  256 rows,
// 32 FP32 matrices: 11 us; a walk over 64-row steps that each read their own tiles took 21 us.
template <typename T>
__global__ __launch_bounds__(1024) void k_solve_small(const T* __restrict__ a, int64_t lda, int n,
                                                      const int32_t* __restrict__ perm, const T* __restrict__ inv,
                                                      T* __restrict__ x, int64_t ldx, int64_t sa, int64_t sx) {
    __shared__ T xs[kSW];
    __shared__ T red[16][kSB];
    __shared__ T yb[kSB];
    const int t = threadIdx.x, r = t & 63, g = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nblk = (n + kSB - 1) / kSB;
    a += (int64_t)blockIdx.z * sa;  // batch: one matrix per blockIdx.z
    inv += (int64_t)blockIdx.z * 2 * nblk * kSB * kSB;
    T* xc = x + (int64_t)blockIdx.z * sx + (int64_t)blockIdx.x * ldx;
    SolveTiles<T, true> lo;
    SolveTiles<T, false> up;
    lo.load(a, lda, n, inv, r, g);
    if (sizeof(T) == 4) up.load(a, lda, n, inv + (int64_t)nblk * kSB * kSB, r, g);
    if (t < kSW) xs[t] = t < n ? xc[perm[(int64_t)blockIdx.z * n + t]] : T(0);
    __syncthreads();
    {
        T acc[4] = {T(0), T(0), T(0), T(0)};
        lo.solve(xs, red, yb, acc, n, t);
    }
    if (sizeof(T) == 8) up.load(a, lda, n, inv + (int64_t)nblk * kSB * kSB, r, g);
    T acc[4] = {T(0), T(0), T(0), T(0)};
    up.solve(xs, red, yb, acc, n, t);
    if (t < n) xc[t] = xs[t];
}

// x = P x, one work-group per right-hand side
template <typename T>
__global__ __launch_bounds__(1024) void k_solve_perm(int n, const int32_t* __restrict__ perm, T* __restrict__ x,
                                                     int64_t ldx, int64_t sx) {
    __shared__ T xs[kSolveMaxN];
    perm += (int64_t)blockIdx.z * n;
    T* xc = x + (int64_t)blockIdx.z * sx + (int64_t)blockIdx.x * ldx;
    for (int i = threadIdx.x; i < n; i += 1024) xs[i] = xc[i];
    __syncthreads();
    for (int i = threadIdx.x; i < n; i += 1024) xc[i] = xs[perm[i]];
}

// Substitution step after the rows of step b (kSW rows, x_b final from the previous launch): work-group 0
// subtracts their part from the next kSW rows in order and finishes these (SolveTiles); work-group j > 0
// subtracts it from the j-th 64-row block beyond.  The first launch of a triangle (b = -1 forward, the number
// of steps backward) only finishes its first rows.  Each off-diagonal tile is read once per right-hand side, 64
// consecutive rows per column by each wave, 16 waves splitting the columns.
// Bound by the chain of launches and, in work-group 0, of its four 64-row solves: all its tiles but the
// inverse's products are read before the chain starts, and 256 rows per launch instead of 64 take a quarter of the
// launches.  Both substitutions of one FP64 right-hand side at n = 4096: 1.04 -> 0.60 ms; FP32 at n = 16384,
// 2 matrices: 5.3 -> 1.9 ms.
template <typename T, bool LOWER>
__global__ __launch_bounds__(1024) void k_trsv_step(const T* __restrict__ a, int64_t lda, int n,
                                                    const T* __restrict__ inv, T* __restrict__ x, int64_t ldx,
                                                    int64_t sa, int64_t sx, int b) {
    __shared__ T xb[kSW];
    __shared__ T xn[kSW];
    __shared__ T red[16][kSB];
    __shared__ T yb[kSB];
    const int t = threadIdx.x, r = t & 63, g = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nblk = (n + kSB - 1) / kSB, nst = (n + kSW - 1) / kSW;
    a += (int64_t)blockIdx.z * sa;
    inv += (int64_t)blockIdx.z * 2 * nblk * kSB * kSB + (LOWER ? 0 : (int64_t)nblk * kSB * kSB);
    T* xc = x + (int64_t)blockIdx.z * sx + (int64_t)blockIdx.y * ldx;
    const int c0 = b * kSW;
    const bool has_b = LOWER ? b >= 0 : b < nst;
    const int cols = has_b ? min(kSW, n - c0) : 0;
    // sum over this thread's 16 columns of step b in row `row` (past the matrix: its last row or column is read, and
    // not used)
    auto part = [&](int row) {
        const unsigned at = min(row, n - 1);
        T m[16];
#pragma unroll
        for (int c = 0; c < 16; c++) m[c] = (a + (int64_t)min(c0 + 16 * g + c, n - 1) * lda)[at];
        T s = T(0);
#pragma unroll
        for (int c = 0; c < 16; c++) s += 16 * g + c < cols ? m[c] * xb[16 * g + c] : T(0);
        return s;
    };
    if (has_b && t < kSW) xb[t] = t < cols ? xc[c0 + t] : T(0);
    if (blockIdx.x > 0) {
        const int j = blockIdx.x - 1;
        const int r0 = LOWER ? (b + 2) * kSW + j * kSB : (b - 1) * kSW - (j + 1) * kSB;
        const T y = t < kSB && r0 + t < n ? xc[r0 + t] : T(0);
        __syncthreads();
        red[g][r] = part(r0 + r);
        __syncthreads();
        if (t < kSB && r0 + t < n) {
            T s = y;
#pragma unroll
            for (int k = 0; k < 16; k++) s -= red[k][t];
            xc[r0 + t] = s;
        }
        return;
    }
    const int w = LOWER ? b + 1 : b - 1, r0 = w * kSW, nr = n - r0;
    SolveTiles<T, LOWER> tiles;
    if (sizeof(T) == 4) tiles.load(a + r0 + (int64_t)r0 * lda, lda, nr, inv + (int64_t)w * 4 * kSB * kSB, r, g);
    if (t < kSW) xn[t] = t < nr ? xc[r0 + t] : T(0);
    __syncthreads();
    T acc[4] = {T(0), T(0), T(0), T(0)};
    if (has_b)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            acc[q] = part(r0 + q * kSB + r);
            __builtin_amdgcn_sched_barrier(0);  // 16 loads in flight beside the tiles: 128 registers hold no more
        }
    if (sizeof(T) == 8) tiles.load(a + r0 + (int64_t)r0 * lda, lda, nr, inv + (int64_t)w * 4 * kSB * kSB, r, g);
    tiles.solve(xn, red, yb, acc, nr, t);
    if (t < min(kSW, nr)) xc[r0 + t] = xn[t];
}

// One work-group per right-hand side, its column in LDS, 64 rows at a time: each off-diagonal row of tiles is
// read where its rows are solved, 64 consecutive rows per column, split over the 16 waves.
template <typename T>
__global__ __launch_bounds__(1024) void k_solve_blocked(const T* __restrict__ a, int64_t lda, int n,
                                                        const int32_t* __restrict__ perm, const T* __restrict__ inv,
                                                        T* __restrict__ x, int64_t ldx, int64_t sa, int64_t sx) {
    __shared__ T xs[kBlockedMaxN];
    __shared__ T red[16][kSB];
    __shared__ T yb[kSB];
    const int t = threadIdx.x, r = t & 63, g = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nblk = (n + kSB - 1) / kSB;
    a += (int64_t)blockIdx.z * sa;  // batch: one matrix per blockIdx.z
    perm += (int64_t)blockIdx.z * n;
    inv += (int64_t)blockIdx.z * 2 * nblk * kSB * kSB;
    T* xc = x + (int64_t)blockIdx.z * sx + (int64_t)blockIdx.x * ldx;
    for (int i = t; i < n; i += 1024) xs[i] = xc[perm[i]];
    __syncthreads();
    for (int e = 0; e < 2 * nblk; e++) {  // L from the first block on, then U from the last
        const bool lower = e < nblk;
        const int b = lower ? e : 2 * nblk - 1 - e;
        const int r0 = b * kSB, rb = min(kSB, n - r0);
        const T* ib = inv + ((int64_t)(lower ? 0 : nblk) + b) * kSB * kSB;
        T acc = T(0);
        if (r < rb)
            for (int j = (lower ? 0 : r0 + kSB) + g; j < (lower ? r0 : n); j += 16)
                acc += a[(r0 + r) + (int64_t)j * lda] * xs[j];
        red[g][r] = acc;
        __syncthreads();
        if (t < kSB) {
            T y = t < rb ? xs[r0 + t] : T(0);
#pragma unroll
            for (int q = 0; q < 16; q++) y -= red[q][t];
            yb[t] = y;
        }
        __syncthreads();
        T s = T(0);
#pragma unroll
        for (int p = 4 * g; p < 4 * g + 4; p++) s += ib[r + p * kSB] * yb[p];
        red[g][r] = s;
        __syncthreads();
        if (t < rb) {
            T v = T(0);
#pragma unroll
            for (int q = 0; q < 16; q++) v += red[q][t];
            xs[r0 + t] = v;
        }
        __syncthreads();
    }
    for (int i = t; i < n; i += 1024) xc[i] = xs[i];
}

// k_trsv_step's substitutions by 64 rows: work-group j subtracts the part of block b's rows from the j-th block
// after it (forward) or before it (backward), group 0 then finishes its block with the inverse.
template <typename T, bool LOWER>
__global__ __launch_bounds__(256) void k_trsv_block(const T* __restrict__ a, int64_t lda, int n,
                                                    const T* __restrict__ inv, T* __restrict__ x, int64_t ldx,
                                                    int64_t sa, int64_t sx, int b) {
    __shared__ T xb[kSB];
    __shared__ T red[4][kSB];
    __shared__ T yb[kSB];
    const int t = threadIdx.x, rl = t & 63, g = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nblk = (n + kSB - 1) / kSB;
    a += (int64_t)blockIdx.z * sa;
    inv += (int64_t)blockIdx.z * 2 * nblk * kSB * kSB + (LOWER ? 0 : (int64_t)nblk * kSB * kSB);
    T* xc = x + (int64_t)blockIdx.z * sx + (int64_t)blockIdx.y * ldx;
    const int j = blockIdx.x;
    const int r = LOWER ? b + 1 + j : b - 1 - j;  // this group's row block
    const int r0 = r * kSB, c0 = b * kSB;
    T y = T(0);
    if (t < kSB) y = r0 + t < n ? xc[r0 + t] : T(0);
    if (LOWER ? b >= 0 : b < nblk) {
        if (t < kSB) xb[t] = c0 + t < n ? xc[c0 + t] : T(0);
        __syncthreads();
        T acc = T(0);
        if (r0 + rl < n) {
            const T* ab = a + (r0 + rl) + (int64_t)c0 * lda;
#pragma unroll 4
            for (int c = 16 * g; c < 16 * g + 16; c++)
                if (c0 + c < n) acc += ab[(int64_t)c * lda] * xb[c];
        }
        red[g][rl] = acc;
        __syncthreads();
        if (t < kSB) y -= red[0][t] + red[1][t] + red[2][t] + red[3][t];
    }
    if (j != 0) {  // a later block: store the partial update
        if (t < kSB && r0 + t < n) xc[r0 + t] = y;
        return;
    }
    // the next block in order: finish it with its diagonal-block inverse
    if (t < kSB) yb[t] = y;
    __syncthreads();
    const T* ib = inv + (int64_t)r * kSB * kSB;
    T s = T(0);
#pragma unroll
    for (int p = 16 * g; p < 16 * g + 16; p++) s += ib[rl + p * kSB] * yb[p];
    red[g][rl] = s;
    __syncthreads();
    if (t < kSB && r0 + t < n) xc[r0 + t] = red[0][t] + red[1][t] + red[2][t] + red[3][t];
}

// X_b = inv X_b for the 64 rows of a diagonal block (rb of them in the matrix) and all right-hand sides, a wave
// per 16 of them, on the matrix cores
template <typename T>
__global__ __launch_bounds__(256) void k_inv_apply(const T* __restrict__ inv, T* __restrict__ x, int64_t ldx, int rb,
                                                   int nrhs) {
    using M = Mf16<T>;
    typedef typename M::vacc vacc;
    const int lane = threadIdx.x & 63, m = lane & 15;
    const int j = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16 + m;
    T* xc = x + (int64_t)min(j, nrhs - 1) * ldx;
    T q[4][4];
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = 16 * k + M::k(lane, r);
            q[k][r] = row < rb ? xc[row] : T(0);
        }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        vacc y = {T(0), T(0), T(0), T(0)};
#pragma unroll
        for (int k = 0; k < 4; k++)
#pragma unroll
            for (int r = 0; r < 4; r++) y = M::mfma(inv[16 * i + m + (16 * k + M::k(lane, r)) * kSB], q[k][r], y);
        if (j < nrhs)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 16 * i + M::k(lane, r);
                if (row < rb) xc[row] = y[r];
            }
    }
}

// How a solve past kSW rows runs.  Each line lies about where the two sides measured alike (us; in brackets n,
// matrices, right-hand sides each):
//   kRouteBlocked, a work-group per right-hand side: a single launch where the steps' chain has two and more per 256
//     rows (FP64 [300, 1, 1]: 63 and 36), and enough work-groups with many right-hand sides (FP64 [600, 1, 96]: 122
//     and 79, [700, 2, 200]: 317 and 169; FP32 [700, 1, 200]: 116 and 77, but [1000, 8, 200]: 939 and 1166);
//   kRouteProducts, 64 rows at a time as products over all right-hand sides of a matrix ([4096, 1, 200]: steps FP64 4015,
//     products 2641; FP32 2413 and 1993);
//   kRouteBlocks, steps of 64 rows: a step of 256 rows and right-hand side holds a work-group of 1024 threads through
//     its serial part, which many right-hand sides queue for (FP64 [4096, 1, 48]: 1434 and 1198, [4096, 1, 24]: 1018
//     and 1059; FP32 [8100, 1, 48]: 3318 and 2934);
//   kRouteSteps otherwise.
// The route, and with it the rounding, depends on the number of matrices only from 8 matrices and 8 right-hand sides
// on: a served request gives the same answer in any batch.
enum SolveRoute { kRouteSteps, kRouteBlocked, kRouteBlocks, kRouteProducts };

template <typename T>
SolveRoute solve_route(int64_t n, int64_t nrhs, int64_t batch) {
    constexpr bool f64 = sizeof(T) == 8;
    const int64_t rows = nrhs * n;
    if (rows >= (n <= 896 ? 1024 : f64 ? 896 : 768) * 1024) return kRouteProducts;
    if (n <= 320) return kRouteBlocked;
    if (n <= kBlockedMaxN) {
        if (nrhs >= (f64 ? (n <= 640 ? 64 : 200) : n <= 512 ? 512 : n <= 896 ? 160 : INT64_MAX)) return kRouteBlocked;
        if (batch >= 8 && nrhs >= 8 && nrhs * batch >= 256 && (f64 || (n > 512 && n <= 896))) return kRouteBlocked;
        return kRouteSteps;
    }
    if (f64 ? rows >= (n < 1400 ? 256 : 128) * 1024 : n >= 3072 && rows >= 376 * 1024) return kRouteBlocks;
    return kRouteSteps;
}

// What getrs makes of the factors before it sees a right-hand side: inverses of the diagonal blocks, the
// composed interchanges, and the lists they come from.
template <typename T>
struct SolvePrep {
    T* inv;
    int32_t *perm, *pairs;
    static bool covers(int64_t n) { return n <= kSolveMaxN; }
    static size_t bytes(int n, int batch) {
        const size_t nblk = (n + kSB - 1) / kSB;
        return (sizeof(T) * 2 * nblk * kSB * kSB + sizeof(int32_t) * (n + nblk * kSolvePairs)) * batch;
    }
    void place(void* ws, int n, int batch) {
        const size_t nblk = (n + kSB - 1) / kSB;
        inv = static_cast<T*>(ws);
        perm = reinterpret_cast<int32_t*>(inv + 2 * nblk * kSB * kSB * batch);
        pairs = perm + (size_t)n * batch;
    }
    int make(const T* a, int64_t lda, int n, int64_t sa, int batch, const int32_t* ipiv, hipStream_t st) const {
        const int nblk = (n + kSB - 1) / kSB;
        hipLaunchKernelGGL(k_solve_prep<T>, dim3(nblk, 3, batch), dim3(256), 0, st, a, lda, n, ipiv, pairs, inv, sa);
        TVLM_LAUNCHED();
        hipLaunchKernelGGL(k_solve_compose, dim3(batch), dim3(256), 0, st, n, pairs, perm);
        TVLM_LAUNCHED();
        return TVLM_OK;
    }
    int solve(const T* a, int64_t lda, int n, int64_t sa, int batch, T* x, int64_t ldx, int64_t sx, int nrhs,
              hipStream_t st) const {
        if (n <= kSW) {
            hipLaunchKernelGGL(k_solve_small<T>, dim3(nrhs, 1, batch), dim3(1024), 0, st, a, lda, n, perm, inv, x, ldx,
                               sa, sx);
            TVLM_LAUNCHED();
            return TVLM_OK;
        }
        SolveRoute route = solve_route<T>(n, nrhs, batch);
        if (route == kRouteProducts && (lda >= kUpdMaxLd || ldx >= kUpdMaxLd)) route = kRouteBlocks;
        if (route == kRouteBlocked) {
            hipLaunchKernelGGL(k_solve_blocked<T>, dim3(nrhs, 1, batch), dim3(1024), 0, st, a, lda, n, perm, inv, x, ldx,
                               sa, sx);
            TVLM_LAUNCHED();
            return TVLM_OK;
        }
        hipLaunchKernelGGL(k_solve_perm<T>, dim3(nrhs, 1, batch), dim3(1024), 0, st, n, perm, x, ldx, sx);
        TVLM_LAUNCHED();
        const int nblk = (n + kSB - 1) / kSB, nst = (n + kSW - 1) / kSW;
        if (route == kRouteBlocks) {
            for (int b = -1; b < nblk - 1; b++) {
                hipLaunchKernelGGL((k_trsv_block<T, true>), dim3(b < 0 ? 1 : nblk - 1 - b, nrhs, batch), dim3(256), 0, st,
                                   a, lda, n, inv, x, ldx, sa, sx, b);
                TVLM_LAUNCHED();
            }
            for (int b = nblk; b > 0; b--) {
                hipLaunchKernelGGL((k_trsv_block<T, false>), dim3(b == nblk ? 1 : b, nrhs, batch), dim3(256), 0, st, a, lda,
                                   n, inv, x, ldx, sa, sx, b);
                TVLM_LAUNCHED();
            }
            return TVLM_OK;
        }
        if (route == kRouteProducts) {
            for (int z = 0; z < batch; z++) {
                const T* az = a + (int64_t)z * sa;
                const T* iz = inv + (int64_t)z * 2 * nblk * kSB * kSB;
                T* xz = x + (int64_t)z * sx;
                auto finish = [&](int b, int tri) {
                    hipLaunchKernelGGL(k_inv_apply<T>, dim3((nrhs + 63) / 64), dim3(256), 0, st,
                                       iz + ((int64_t)tri * nblk + b) * kSB * kSB, xz + b * kSB, ldx,
                                       n - b * kSB < kSB ? n - b * kSB : kSB, nrhs);
                };
                for (int b = 0; b < nblk; b++) {
                    const int c0 = b * kSB, r0 = c0 + kSB;
                    finish(b, 0);
                    TVLM_LAUNCHED();
                    launch_update<T>(xz + r0, ldx, az + r0 + (int64_t)c0 * lda, lda, xz + c0, ldx, n - r0, nrhs, kSB, 0, 1,
                                     st);
                    TVLM_LAUNCHED();
                }
                for (int b = nblk - 1; b >= 0; b--) {
                    const int c0 = b * kSB;
                    finish(b, 1);
                    TVLM_LAUNCHED();
                    launch_update<T>(xz, ldx, az + (int64_t)c0 * lda, lda, xz + c0, ldx, c0, nrhs,
                                     n - c0 < kSB ? n - c0 : kSB, 0, 1, st);
                    TVLM_LAUNCHED();
                }
            }
            return TVLM_OK;
        }
        for (int b = -1; b < nst - 1; b++) {
            const int beyond = b < 0 ? 0 : nblk - 4 * (b + 2);
            hipLaunchKernelGGL((k_trsv_step<T, true>), dim3(1 + (beyond > 0 ? beyond : 0), nrhs, batch), dim3(1024), 0, st,
                               a, lda, n, inv, x, ldx, sa, sx, b);
            TVLM_LAUNCHED();
        }
        for (int b = nst; b > 0; b--) {
            const int beyond = b == nst ? 0 : 4 * (b - 1);
            hipLaunchKernelGGL((k_trsv_step<T, false>), dim3(1 + beyond, nrhs, batch), dim3(1024), 0, st, a, lda, n, inv, x,
                               ldx, sa, sx, b);
            TVLM_LAUNCHED();
        }
        return TVLM_OK;
    }
};

// shape[2] > 1 solves a batch: matrix b at A.ptr + b A.stride[2] with pivots ipiv + b n, its
// right-hand sides at X.ptr + b X.stride[2].  prepared: the batch's SolvePrep, made from these factors.
template <typename T>
int getrs(const tvlm_view* av, const int32_t* ipiv, const tvlm_view* xv, void* stream, void* prepared = nullptr) {
    TVLM_REQUIRE(av && xv && av->ptr && xv->ptr && ipiv, "null argument");
    TVLM_REQUIRE(av->stride[0] == 1 && xv->stride[0] == 1, "column-major operands required");
    const int n = (int)av->shape[0];
    TVLM_REQUIRE(av->shape[1] == n && xv->shape[0] == n, "shape mismatch");
    const int batch = (int)av->shape[2];
    TVLM_REQUIRE(xv->shape[2] == batch, "A has %d matrices, X %lld right-hand-side sets", batch,
                 (long long)xv->shape[2]);
    TVLM_REQUIRE(batch >= 1 && batch <= 65535, "batch %d out of range", batch);
    const int nrhs = (int)xv->shape[1];
    if (n == 0 || nrhs == 0) return TVLM_OK;
    const int64_t lda = av->stride[1], ldx = nrhs > 1 ? xv->stride[1] : n;
    const int64_t sa = av->stride[2], sx = xv->stride[2];
    hipStream_t st = as_stream(stream);
    const T* a = static_cast<const T*>(av->ptr);
    T* x = static_cast<T*>(xv->ptr);
    if (SolvePrep<T>::covers(n)) {
        SolvePrep<T> P;
        void* ws = prepared;
        if (!ws) TVLM_TRY(device_workspace(SolvePrep<T>::bytes(n, batch), &ws, kWsSolveInv, st));
        P.place(ws, n, batch);
        if (!prepared) TVLM_TRY(P.make(a, lda, n, sa, batch, ipiv, st));
        return P.solve(a, lda, n, sa, batch, x, ldx, sx, nrhs, st);
    }
    for (int z = 0; z < batch; z++) {
        const T* az = a + (int64_t)z * sa;
        const int32_t* pz = ipiv + (int64_t)z * n;
        T* xz = x + (int64_t)z * sx;
        hipLaunchKernelGGL(k_apply_pivots<T>, dim3(nrhs), dim3(64), 0, st, xz, ldx, n, pz);
        TVLM_LAUNCHED();
        for (int r0 = 0; r0 < n; r0 += SB) {  // forward: L
            const int nb = (n - r0 < SB) ? n - r0 : SB;
            hipLaunchKernelGGL((k_diag_solve<T, true>), dim3(nrhs), dim3(SB), 0, st, az, lda, r0, nb, xz, ldx);
            TVLM_LAUNCHED();
            if (r0 + nb < n) {
                hipLaunchKernelGGL(k_off_update<T>, dim3((n - r0 - nb + 255) / 256, nrhs), dim3(256), 0, st, az, lda,
                                   r0 + nb, n, r0, nb, xz, ldx);
                TVLM_LAUNCHED();
            }
        }
        const int nblk = (n + SB - 1) / SB;
        for (int b = nblk - 1; b >= 0; b--) {  // backward: U
            const int r0 = b * SB;
            const int nb = (n - r0 < SB) ? n - r0 : SB;
            hipLaunchKernelGGL((k_diag_solve<T, false>), dim3(nrhs), dim3(SB), 0, st, az, lda, r0, nb, xz, ldx);
            TVLM_LAUNCHED();
            if (r0 > 0) {
                hipLaunchKernelGGL(k_off_update<T>, dim3((r0 + 255) / 256, nrhs), dim3(256), 0, st, az, lda, 0, r0, r0,
                                   nb, xz, ldx);
                TVLM_LAUNCHED();
            }
        }
    }
    return TVLM_OK;
}

}  // namespace

void release_lu_stream(hipStream_t stream) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return;
    LookaheadStreams L;
    {
        std::lock_guard<std::mutex> lock(g_lookahead_mu);
        auto it = g_lookahead.find(std::make_pair(dev, stream));
        if (it == g_lookahead.end()) return;
        L = it->second;
        g_lookahead.erase(it);
    }
    if (L.side) {
        (void)hipStreamSynchronize(L.side);
        (void)hipStreamDestroy(L.side);
    }
    if (L.narrow_done) (void)hipEventDestroy(L.narrow_done);
    if (L.rest_done) (void)hipEventDestroy(L.rest_done);
}

int getrf_single_group_f64(const tvlm_view* a, int32_t* ipiv, int32_t* info, void* stream) {
    return getrf<double>(a, ipiv, info, stream, false);
}
int getrf_single_group_f32(const tvlm_view* a, int32_t* ipiv, int32_t* info, void* stream) {
    return getrf<float>(a, ipiv, info, stream, false);
}

size_t getrs_prep_bytes_f32(int64_t n, int batch) {
    return SolvePrep<float>::covers(n) ? SolvePrep<float>::bytes((int)n, batch) : 0;
}
int getrs_prepare_f32(const tvlm_view* a, const int32_t* ipiv, void* prep, hipStream_t st) {
    if (!prep) return TVLM_OK;
    SolvePrep<float> P;
    P.place(prep, (int)a->shape[0], (int)a->shape[2]);
    return P.make(static_cast<const float*>(a->ptr), a->stride[1], (int)a->shape[0], a->stride[2], (int)a->shape[2], ipiv,
                  st);
}
int getrs_prepared_f32(const tvlm_view* a, const int32_t* ipiv, void* prep, const tvlm_view* x, hipStream_t st) {
    return getrs<float>(a, ipiv, x, st, prep);
}

}  // namespace tvlm

extern "C" {
int tvlm_getrf_plan(int64_t n, int32_t batch, int32_t elem_bytes, int32_t* path, int32_t* n_steps, int32_t* groups,
                    int32_t* ctr_set, int32_t max_steps, int64_t* coop_ws_bytes) {
    TVLM_REQUIRE(path && n_steps, "null argument");
    TVLM_REQUIRE(n >= 0 && n <= (int64_t)1 << 30 && batch >= 1 && batch <= 65535, "n %lld / batch %d out of range",
                 (long long)n, batch);
    TVLM_REQUIRE(elem_bytes == 4 || elem_bytes == 8, "elem_bytes must be 4 or 8");
    const tvlm::GetrfPlan P = elem_bytes == 8 ? tvlm::getrf_plan<double>((int)n, batch, true)
                                              : tvlm::getrf_plan<float>((int)n, batch, true);
    *path = P.path;
    *n_steps = (int32_t)P.steps.size();
    if (coop_ws_bytes) *coop_ws_bytes = (int64_t)P.coop_bytes((size_t)elem_bytes);
    if (groups || ctr_set) {
        TVLM_REQUIRE((int64_t)P.steps.size() <= (int64_t)max_steps, "%zu panels, room for %d", P.steps.size(), max_steps);
        for (size_t k = 0; k < P.steps.size(); k++) {
            if (groups) groups[k] = P.steps[k].groups;
            if (ctr_set) ctr_set[k] = P.steps[k].ctr_set;
        }
    }
    return TVLM_OK;
}
int tvlm_lu_update(int32_t elem_bytes, void* c, int64_t ldc, const void* a, int64_t lda, const void* b, int64_t ldb,
                   int64_t m, int64_t n, int64_t k, int32_t batch, int64_t stride, void* stream) {
    TVLM_REQUIRE(elem_bytes == 4 || elem_bytes == 8, "elem_bytes must be 4 or 8");
    TVLM_REQUIRE(m >= 0 && n >= 0 && k >= 0 && m < (1 << 30) && n < (1 << 30) && k < (1 << 30), "m/n/k out of range");
    TVLM_REQUIRE(batch >= 1 && batch <= 65535 && (batch == 1 || stride >= 0), "batch %d / stride out of range", batch);
    TVLM_REQUIRE(ldc >= (m > 1 ? m : 1) && lda >= (m > 1 ? m : 1) && ldb >= (k > 1 ? k : 1) &&
                     ldc < tvlm::kUpdMaxLd && lda < tvlm::kUpdMaxLd && ldb < tvlm::kUpdMaxLd,
                 "leading dimensions out of range");
    if (m == 0 || n == 0 || k == 0) return TVLM_OK;
    TVLM_REQUIRE(c && a && b, "null matrix");
    const hipStream_t st = (hipStream_t)stream;
    if (elem_bytes == 8)
        tvlm::launch_update<double>((double*)c, ldc, (const double*)a, lda, (const double*)b, ldb, (int)m, (int)n, (int)k,
                                    stride, batch, st);
    else
        tvlm::launch_update<float>((float*)c, ldc, (const float*)a, lda, (const float*)b, ldb, (int)m, (int)n, (int)k,
                                   stride, batch, st);
    TVLM_LAUNCHED();
    return TVLM_OK;
}
int tvlm_lu_set_coop_spin_limit(uint32_t limit) {
    tvlm::g_coop_spin_limit.store(limit == 0 ? tvlm::kCoopSpinLimit : limit);
    return TVLM_OK;
}
int tvlm_getrf_f64(const tvlm_view* a, int32_t* ipiv, int32_t* info, void* stream) {
    return tvlm::getrf<double>(a, ipiv, info, stream);
}
int tvlm_getrf_f32(const tvlm_view* a, int32_t* ipiv, int32_t* info, void* stream) {
    return tvlm::getrf<float>(a, ipiv, info, stream);
}
int tvlm_getrs_f64(const tvlm_view* a, const int32_t* ipiv, const tvlm_view* x, void* stream) {
    return tvlm::getrs<double>(a, ipiv, x, stream);
}
int tvlm_getrs_f32(const tvlm_view* a, const int32_t* ipiv, const tvlm_view* x, void* stream) {
    return tvlm::getrs<float>(a, ipiv, x, stream);
}
}
