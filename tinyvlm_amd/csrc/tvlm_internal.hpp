// tvlm_internal.hpp -- shared device/host helpers of the gfx950 backend.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>

#include "../../include/tinyvlm_hip.h"

namespace tvlm {

// ---- error reporting --------------------------------------------------------------------------
void set_error(const char* fmt, ...);

#define TVLM_HIP(expr)                                                                              \
    do {                                                                                            \
        hipError_t e_ = (expr);                                                                     \
        if (e_ != hipSuccess) {                                                                     \
            ::tvlm::set_error("%s failed: %s (%s:%d)", #expr, hipGetErrorString(e_), __FILE__,      \
                              __LINE__);                                                            \
            return e_ == hipErrorOutOfMemory ? TVLM_ERR_NOMEM : TVLM_ERR_HIP;                       \
        }                                                                                           \
    } while (0)

#define TVLM_REQUIRE(cond, ...)                                                                     \
    do {                                                                                            \
        if (!(cond)) {                                                                              \
            ::tvlm::set_error(__VA_ARGS__);                                                         \
            return TVLM_ERR_INVALID;                                                                \
        }                                                                                           \
    } while (0)

#define TVLM_TRY(expr)                                                                              \
    do {                                                                                            \
        int s_ = (expr);                                                                            \
        if (s_ != TVLM_OK) return s_;                                                               \
    } while (0)

#define TVLM_LAUNCHED() TVLM_HIP(hipGetLastError())

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// ---- view validation --------------------------------------------------------------------------
// 3-D per-surface tensors {a, b, k} must be "plane contiguous": stride[0] == 1 and
// stride[1] == shape[0] (what the reference kernels assume, vlm_backend_cpu.cpp:111, :202).
inline bool plane_contiguous(const tvlm_view& v) {
    return v.ptr != nullptr && v.stride[0] == 1 && v.stride[1] == v.shape[0];
}

// Scratch buffers owned by the library (grow-only), one per device, slot and stream: wake-induction
// tile partials, LU row-interchange lists, triangular-solve block inverses, the exchange buffers of
// the cooperative LU panels, the speculative panels' results.  Work queued on different streams never shares a buffer, so concurrent
// solves on separate streams are safe; work on one stream is ordered by the stream.
enum WorkspaceSlot { kWsWakePartials = 0, kWsLuPerm = 1, kWsSolveInv = 2, kWsLuCoop = 3, kWsLsq = 4, kWsLuSpec = 5,
                     kWorkspaceSlots = 6 };
int device_workspace(size_t bytes, void** out, int slot, hipStream_t stream);
// Frees what the library keeps for one stream on the current device (its scratch buffers, its
// rocBLAS handle, its look-ahead side stream); the stream's work must have finished.
void release_workspaces(hipStream_t stream);
void release_lu_stream(hipStream_t stream);

// A stream with a hardware queue of its own: created with an all-CUs mask (streams created
// without a mask share a small pool of queues, and two streams on one queue run one after the
// other).  Default priority.
int create_queue_stream(hipStream_t* out);

// Looks up the device address of the allocation-free wake induction's fixed scratch array on the
// current device (once per device; tvlm_init calls it so that later calls find it set up).
int noalloc_scratch_setup();

// getrf with every panel in one work-group (no cooperative panels, hence no waits between
// work-groups): the recovery path after a cooperative panel's bounded wait gave up
int getrf_single_group_f64(const tvlm_view* a, int32_t* ipiv, int32_t* info, void* stream);
int getrf_single_group_f32(const tvlm_view* a, int32_t* ipiv, int32_t* info, void* stream);

// getrs of several right-hand sides one after another on the same factors: what it derives from them first
// (block inverses, composed interchanges) is made once, in `prep` of getrs_prep_bytes_f32 bytes (0 where n is
// past the sizes that use it; prep is then null), for as long as the factors stand.
size_t getrs_prep_bytes_f32(int64_t n, int batch);
int getrs_prepare_f32(const tvlm_view* a, const int32_t* ipiv, void* prep, hipStream_t stream);
int getrs_prepared_f32(const tvlm_view* a, const int32_t* ipiv, void* prep, const tvlm_view* x, hipStream_t stream);

constexpr int32_t kGetrfStalled = -999;  // info of a matrix whose cooperative panel gave up waiting

// Work-group targets of the wake-induction launches, library-wide (tvlm_set_tile_targets): the
// Backend form's tile shape (wake_tile_shape) and new UVLM plans' lattice launches.
constexpr int kTargetGroups = 2048;     // default of wake_target_groups()
constexpr int kLatTargetGroups = 1024;  // default of lattice_target_groups()
int wake_target_groups();
int lattice_target_groups();

// lhs_assemble in the FP64 seeded form (the served steady solve uses it; exported as
// tvlm_lhs_assemble_seeded_f64)
int lhs_assemble_seeded_f64(const tvlm_view* lhs, int32_t n_surf, const tvlm_view* colloc, const tvlm_view* normals,
                            const tvlm_view* verts_wing, const tvlm_view* verts_wake, int32_t iteration, void* stream);

// Grouped assembly in the FP64 seeded form that sets the matrices (of the group's first n_items items)
// instead of adding to them, and stores them rounded to FP32 as well: element k past base64 at base32 + k.
int lhs_group_assign_seeded(tvlm_lhs_group* group, int32_t n_items, const double* base64, float* base32,
                            hipStream_t stream);

// ---- small vector type ------------------------------------------------------------------------
template <typename T>
struct v3 {
    T x, y, z;
};
template <typename T>
__host__ __device__ inline v3<T> operator-(const v3<T>& a, const v3<T>& b) {
    return {a.x - b.x, a.y - b.y, a.z - b.z};
}
template <typename T>
__host__ __device__ inline v3<T> operator+(const v3<T>& a, const v3<T>& b) {
    return {a.x + b.x, a.y + b.y, a.z + b.z};
}
template <typename T>
__host__ __device__ inline v3<T> operator*(T s, const v3<T>& a) {
    return {s * a.x, s * a.y, s * a.z};
}
template <typename T>
__host__ __device__ inline T dot(const v3<T>& a, const v3<T>& b) {
    return a.x * b.x + a.y * b.y + a.z * b.z;
}
template <typename T>
__host__ __device__ inline v3<T> cross(const v3<T>& a, const v3<T>& b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// ---- Biot-Savart constants (vlm_backend_cpu_kernels.ispc:9-12, :80, :87, :393, :400) -----------
template <typename T>
struct BS;
template <>
struct BS<double> {
    static constexpr double fourpi = (double)(4.0f * 3.141593f);  // the float product 4.0f*PI_f
    static constexpr double cut_cross = (double)1e-10f;            // RCUT
    static constexpr double cut_norm = (double)1e-10f;             // FP64 uses RCUT for the norms too
};
template <>
struct BS<float> {
    static constexpr float fourpi = 4.0f * 3.141593f;
    static constexpr float cut_cross = 1e-10f;  // RCUT on |r1 x r2|^2
    static constexpr float cut_norm = 1e-5f;    // RCUT2 on |r1|, |r2|
};

// ---- panel metrics (vlm_backend_cpu.cpp:391-433, vlm_backend_cpud.cpp:258-300) -----------------
// Normal normalize((v3-v1) x (v2-v0)); area 0.5(|f x b| + |b x e|); collocation point
// 0.5(v0+v1) + k * 0.5(v2+v3-v0-v1), k = 1/2 below EPS_f else alpha / (2 (sin alpha + EPS_f)).
template <typename T>
__device__ __forceinline__ void panel_metrics(T alpha, const v3<T>& v0, const v3<T>& v1, const v3<T>& v2,
                                              const v3<T>& v3_, v3<T>& colloc, v3<T>& normal, T& area) {
    const v3<T> nv = cross(v3_ - v1, v2 - v0);
    const T l = sqrt(dot(nv, nv));
    normal = {nv.x / l, nv.y / l, nv.z / l};
    const v3<T> f = v3_ - v0, b = v2 - v0, e = v1 - v0;
    const v3<T> fb = cross(f, b), be = cross(b, e);
    area = T(0.5) * (sqrt(dot(fb, fb)) + sqrt(dot(be, be)));
    const T eps = (T)1.19209e-07f;  // EPS_f (vlm_types.hpp:24) in both precisions
    const T factor = (alpha < eps) ? T(0.5) : T(0.5) * (alpha / (sin(alpha) + eps));
    const v3<T> chord = T(0.5) * (((v2 + v3_) - v0) - v1);
    colloc = T(0.5) * (v0 + v1) + factor * chord;
}

// One homogeneous point times a column-major 4x4 (row r of verts {P,4} * T^T, vlm_backend.cpp:59-67).
template <typename T>
__device__ __forceinline__ T displace_row(const T* M, int64_t m0, int64_t m1, int r, const T* x) {
    T s = x[0] * M[r * m0 + 0 * m1];
    s += x[1] * M[r * m0 + 1 * m1];
    s += x[2] * M[r * m0 + 2 * m1];
    s += x[3] * M[r * m0 + 3 * m1];
    return s;
}

// ---- FP64 seeded form ---------------------------------------------------------------------------
// FP64 arithmetic throughout, but 1/sqrt and 1/x from the hardware estimates (v_rsq_f64,
// v_rcp_f64) refined by one Newton step in FP64 instead of the multi-instruction correctly rounded
// FP64 sqrt and division (the Newton step squares the estimate's relative error).  MI355X runs
// FP64 add/mul/fma at the rate of non-packed FP32, so this costs about what the FP32 form costs
// while keeping FP64 accuracy.  Cutoffs as the FP64 reference: |r| < RCUT <=> |r|^2 < RCUT^2.
__device__ __forceinline__ double rsqrt_seeded(double x) {
    const double y = __builtin_amdgcn_rsq(x);  // v_rsq_f64 estimate
    return y * (1.5 - 0.5 * x * y * y);
}
__device__ __forceinline__ double rcp_seeded(double x) {
    const double y = __builtin_amdgcn_rcp(x);  // v_rcp_f64 estimate
    return y * (2.0 - x * y);
}

}  // namespace tvlm
