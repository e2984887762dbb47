// tvlm_kernels.hpp -- Biot-Savart assembly kernels shared by the Backend entry points and the
// device-resident solver loops.
//
// lhs block: a work-group owns 64 receivers (one per lane, colloc + normal in registers) and a tile of
// rings (a few chordwise rows x some spans) whose vertices are staged in LDS; its 4 waves split the
// spans and walk them column by column, every segment and vertex of the tile once, reading LDS as a
// broadcast and writing one coalesced 64-element column segment per ring.
//
// wake partials: the wake rings are cut into tiles of rows x spans; a work-group stages one tile's vertex
// rows and circulations in LDS, each wave walks a quarter of its spans for the work-group's 64
// receivers, and the 4 waves reduce in LDS to one partial per (tile, receiver).
// k_wake_reduce then sums the partials of all tiles in a fixed order (bitwise reproducible).
#pragma once

#include "tvlm_internal.hpp"

namespace tvlm {
namespace {

constexpr int kRecv = 64;      // receivers per work-group (one per lane)
constexpr int kWaves = 4;      // waves per work-group
constexpr int kThreads = kRecv * kWaves;

template <typename T>
struct RingSource {
    const T* verts;   // {ns+1, nc+1, 4} plane contiguous
    int64_t vs2;      // plane stride of verts
    int32_t ns, nc;   // panels spanwise / chordwise of the ring surface
    const T* wake;    // {ns+1, nwv, 4} plane contiguous (TE columns only)
    int64_t ws2;
    int32_t nwv;
    int32_t iteration;
};

template <typename T>
struct Receivers {
    const T* colloc;  // {ns, nc, 3}: element p + k*cs2
    int64_t cs2;
    const T* normals;
    int64_t ns2;
    int32_t m;        // number of receivers (panels)
};

// One straight segment a -> b for the receiver and its mirror image in y = 0, in the form selected by
// MODE: 0 exact (sigma = 0), 1 exact with core, 2 FP32 rsqrt form, 3 FP64 seeded form.  The velocity is
// k (crx, cry, crz) + km (mrx, -cry, mrz); both images share the y part of r1 x r2.  Vertex<> holds the
// receiver-relative terms of a vertex, so that the segments meeting there share them, and a ring of
// a lattice shares its segments with its neighbours: per ring about 2.25 segments and 1.25 vertices
// instead of 4 and 4, every term as in the reference (kernels.ispc:69-102, :382-415).  Contraction is
// spelled out: a segment's value must not depend on the kernel it is compiled into (the matrices of a
// grouped launch equal the single ones bit for bit).
template <typename T, int MODE>
struct SegForm {
    struct Vertex {
        T x, y, z, ym;  // c - v, y of the image receiver
        T n, nm;        // MODE 0, 1: |c - v| and the image's; 2, 3: their reciprocals
    };
    struct Seg {
        T k, km, crx, cry, crz, mrx, mrz;
    };
    static __device__ __forceinline__ double fma_(double a, double b, double c) { return __builtin_fma(a, b, c); }
    static __device__ __forceinline__ float fma_(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
    // whether a vertex of this n lies outside the cutoff radius
    static __device__ __forceinline__ bool clear(T n) {
        if constexpr (MODE <= 1)
            return !(n < BS<T>::cut_norm);
        else
            return n <= T(1) / BS<T>::cut_norm;
    }
    static __device__ __forceinline__ Vertex vertex(const v3<T>& c, const T* v) {
#pragma clang fp contract(off)
        Vertex f;
        f.x = c.x - v[0];
        f.y = c.y - v[1];
        f.z = c.z - v[2];
        f.ym = -c.y - v[1];
        const T xz = fma_(f.z, f.z, f.x * f.x);
        const T r2 = fma_(f.y, f.y, xz), r2m = fma_(f.ym, f.ym, xz);
        if constexpr (MODE <= 1) {
            f.n = sqrt(r2);
            f.nm = sqrt(r2m);
        } else {
            if constexpr (MODE == 2) {
                f.n = __builtin_amdgcn_rsqf(r2);
                f.nm = __builtin_amdgcn_rsqf(r2m);
            } else {
                f.n = rsqrt_seeded(r2);
                f.nm = rsqrt_seeded(r2m);
            }
        }
        return f;
    }
    // r0 = b - a
    static __device__ __forceinline__ Seg segment(const Vertex& a, const Vertex& b, const v3<T>& r0, T sigma) {
#pragma clang fp contract(off)
        Seg s;
        s.cry = fma_(a.z, b.x, -(a.x * b.z));
        s.crx = fma_(a.y, b.z, -(a.z * b.y));
        s.crz = fma_(a.x, b.y, -(a.y * b.x));
        s.mrx = fma_(a.ym, b.z, -(a.z * b.ym));
        s.mrz = fma_(a.x, b.ym, -(a.ym * b.x));
        const T cry2 = s.cry * s.cry;
        const T sq = fma_(s.crx, s.crx, fma_(s.crz, s.crz, cry2)), sqm = fma_(s.mrx, s.mrx, fma_(s.mrz, s.mrz, cry2));
        const T d1xz = fma_(r0.z, a.z, r0.x * a.x), d2xz = fma_(r0.z, b.z, r0.x * b.x);
        const T d1 = fma_(r0.y, a.y, d1xz), d2 = fma_(r0.y, b.y, d2xz);
        const T d1m = fma_(r0.y, a.ym, d1xz), d2m = fma_(r0.y, b.ym, d2xz);
        const bool ok = clear(a.n) & clear(b.n), okm = clear(a.nm) & clear(b.nm);
        if constexpr (MODE <= 1) {
            T core = sq, corem = sqm;
            if constexpr (MODE == 1) {
                const T sm = sigma * sigma * fma_(r0.z, r0.z, fma_(r0.y, r0.y, r0.x * r0.x));
                core = sqrt(fma_(sm, sm, sq * sq));
                corem = sqrt(fma_(sm, sm, sqm * sqm));
            }
            const T k = fma_(d1, b.n, -(d2 * a.n)) / (BS<T>::fourpi * core * a.n * b.n);
            const T km = fma_(d1m, b.nm, -(d2m * a.nm)) / (BS<T>::fourpi * corem * a.nm * b.nm);
            s.k = (ok & !(sq < BS<T>::cut_cross)) ? k : T(0);
            s.km = (okm & !(sqm < BS<T>::cut_cross)) ? km : T(0);
        } else {
            T i, im;
            if constexpr (MODE == 2) {
                i = __builtin_amdgcn_rcpf(BS<T>::fourpi * sq);
                im = __builtin_amdgcn_rcpf(BS<T>::fourpi * sqm);
            } else {
                i = rcp_seeded(BS<T>::fourpi * sq);
                im = rcp_seeded(BS<T>::fourpi * sqm);
            }
            s.k = (ok & (sq >= BS<T>::cut_cross)) ? fma_(d1, a.n, -(d2 * b.n)) * i : T(0);
            s.km = (okm & (sqm >= BS<T>::cut_cross)) ? fma_(d1m, a.nm, -(d2m * b.nm)) * im : T(0);
        }
        return s;
    }
    static __device__ __forceinline__ Seg segment(const Vertex& a, const Vertex& b, const T* va, const T* vb, T sigma) {
        return segment(a, b, v3<T>{vb[0] - va[0], vb[1] - va[1], vb[2] - va[2]}, sigma);
    }
    static __device__ __forceinline__ T dot_normal(const Seg& s, const v3<T>& n) {
#pragma clang fp contract(off)
        const T yn = s.cry * n.y;
        return fma_(s.k, fma_(s.crz, n.z, fma_(s.crx, n.x, yn)), s.km * fma_(s.mrz, n.z, fma_(s.mrx, n.x, -yn)));
    }
};

constexpr int kLhsSpans = 16;  // most spans of one wave in an lhs tile

// Shape of the lhs tiles of a (receiver surface, ring surface) pair: rh ring rows and spans per wave,
// the largest that still gives about four work-groups per CU (a tile shares the segments inside it; a
// small matrix needs the waves more).  It depends on the section alone, and a ring's value does not depend
// on the shape.
inline void lhs_tile_shape(int m, int ns, int nc, int& rh, int& spans) {
    constexpr int shapes[][2] = {{4, 16}, {4, 8}, {4, 4}, {2, 4}, {2, 2}, {1, 2}, {1, 1}};
    for (const auto& sh : shapes) {
        rh = sh[0];
        spans = sh[1];
        const int64_t groups =
            (int64_t)((m + kRecv - 1) / kRecv) * ((ns + kWaves * spans - 1) / (kWaves * spans)) * ((nc + rh - 1) / rh);
        if (groups >= 1024) return;
    }
}

// Adds the normal velocity of the lattice's unit rings over one wave's spans [sa, sb) of a staged tile
// (vertex rows 0..rhe, vw columns) to out: ring (q, s) at out[s ld + q lq], or with SUM the rows' rings one
// after another to out[s ld].  A column's old values are read before its rings are computed (set: they
// are 0, except with SUM).  out32, when not null: the same elements rounded to FP32.
template <typename T, int RH, int MODE, bool SUM>
__device__ __forceinline__ void lhs_walk(const T* sv, int vw, int rhe, int sa, int sb, const v3<T>& c, const v3<T>& n,
                                         T sigma, T* __restrict__ out, int64_t ld, int64_t lq, bool set,
                                         float* __restrict__ out32) {
    using S = SegForm<T, MODE>;
    constexpr int NO = SUM ? 1 : RH;
    typename S::Vertex prev[RH + 1];
    T left[RH];
#pragma unroll
    for (int q = 0; q <= RH; q++)
        if (q <= rhe) prev[q] = S::vertex(c, sv + 3 * (q * vw + sa));
#pragma unroll
    for (int q = 0; q < RH; q++)
        if (q < rhe)
            left[q] = S::dot_normal(
                S::segment(prev[q], prev[q + 1], sv + 3 * (q * vw + sa), sv + 3 * ((q + 1) * vw + sa), sigma), n);
#pragma unroll 1
    for (int s = sa; s < sb; s++) {
        T* o = out + s * ld;
        T old[NO];
#pragma unroll
        for (int q = 0; q < NO; q++)
            if (q < rhe) old[q] = set && !SUM ? T(0) : o[q * lq];
        T above = T(0);  // spanwise segment of vertex row q
        typename S::Vertex up{};  // vertex (q, s + 1)
#pragma unroll
        for (int q = 0; q <= RH; q++) {
            if (q <= rhe) {
                const T *va = sv + 3 * (q * vw + s), *vb = va + 3;
                const typename S::Vertex cur = S::vertex(c, vb);
                const T span = S::dot_normal(S::segment(prev[q], cur, va, vb, sigma), n);
                if (q > 0) {
                    const T right = S::dot_normal(S::segment(up, cur, vb - 3 * vw, vb, sigma), n);
                    const T ring = ((above + right) - span) - left[q > 0 ? q - 1 : 0];
                    left[q > 0 ? q - 1 : 0] = right;
                    if constexpr (SUM)
                        old[0] += ring;
                    else {
                        const T v = old[q > 0 ? q - 1 : 0] + ring;
                        o[(q - 1) * lq] = v;
                        if (out32) out32[s * ld + (q - 1) * lq] = (float)v;
                    }
                }
                above = span;
                up = cur;
                prev[q] = cur;
            }
        }
        if constexpr (SUM) {
            o[0] = old[0];
            if (out32) out32[s * ld] = (float)old[0];
        }
    }
}

// One tile of the lhs block of a (receiver surface, ring surface) pair: receivers [bx kRecv, +kRecv)
// x rings of RH rows and kWaves * spans spans.  lhs points at (offset_i, offset_j).  Every thread of the
// work-group calls it (it holds barriers); sv is the caller's LDS staging.
// Bound by VALU issue (exact FP64: two IEEE divisions per segment and image pair).  Ring by ring -> shared
// segments: 16 x 16 wing exact FP64 19.8 -> 12.9 us for a call with its fill (32 -> 256 work-groups), elliptic
// 64 x 64 FP32 113.5 -> 79.5 us, the served batch of 32 of them 60.5 -> 52.2 ms.  With `set` the elements are
// stored without a read, and as FP32 too: that batch 52.2 -> 47.6 ms (no fill, no conversion pass).
template <typename T, int RH, int MODE>  // MODE as SegForm
__device__ __forceinline__ void lhs_tile(T* sv, T* __restrict__ lhs, int64_t ld, const Receivers<T>& rc,
                                         const RingSource<T>& src, T sigma, int bx, int by, int spans, bool set = false,
                                         float* lhs32 = nullptr) {
    const int ns = src.ns, sw = kWaves * spans, tiles_span = (ns + sw - 1) / sw;
    const int s0 = (by % tiles_span) * sw, r0 = (by / tiles_span) * RH;
    const int swe = min(sw, ns - s0), rhe = min(RH, src.nc - r0), vw = swe + 1;
    auto stage = [&](const T* grid, int64_t s2, int row, int rows) {  // vertex rows row .. row + rows
        for (int e = threadIdx.x; e < (rows + 1) * vw; e += kThreads) {
            const T* g = grid + (int64_t)(row + e / vw) * (ns + 1) + s0 + e % vw;
            sv[3 * e + 0] = g[0];
            sv[3 * e + 1] = g[s2];
            sv[3 * e + 2] = g[2 * s2];
        }
    };
    stage(src.verts, src.vs2, r0, rhe);
    __syncthreads();
    const int lane = threadIdx.x & (kRecv - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kRecv);
    const int i = bx * kRecv + lane;
    const bool mine = i < rc.m;
    v3<T> c{}, n{};
    if (mine) {
        c = {rc.colloc[i], rc.colloc[i + rc.cs2], rc.colloc[i + 2 * rc.cs2]};
        n = {rc.normals[i], rc.normals[i + rc.ns2], rc.normals[i + 2 * rc.ns2]};
    }
    const int sa = wave * spans, sb = min(swe, sa + spans);
    T* out = lhs + i + (int64_t)s0 * ld;
    float* out32 = lhs32 ? lhs32 + i + (int64_t)s0 * ld : nullptr;
    if (mine && sa < sb)
        lhs_walk<T, RH, MODE, false>(sv, vw, rhe, sa, sb, c, n, sigma, out + (int64_t)r0 * ns * ld, ld, ns * ld, set,
                                         out32 ? out32 + (int64_t)r0 * ns * ld : nullptr);
    if (src.iteration <= 0 || r0 + rhe < src.nc) return;
    // trailing-edge columns: wake rings of rows nwv-2-k, k < iteration (vlm_backend_cpu.cpp:121-139)
    for (int row = src.nwv - 1 - src.iteration; row < src.nwv - 1; row += RH) {
        const int rows = min(RH, src.nwv - 1 - row);
        __syncthreads();
        stage(src.wake, src.ws2, row, rows);
        __syncthreads();
        if (mine && sa < sb)
            lhs_walk<T, RH, MODE, true>(sv, vw, rows, sa, sb, c, n, sigma, out + (int64_t)(src.nc - 1) * ns * ld, ld, 0,
                                        set, out32 ? out32 + (int64_t)(src.nc - 1) * ns * ld : nullptr);
    }
}

template <int RH>
constexpr int lhs_stage_values() {
    return 3 * (RH + 1) * (kWaves * kLhsSpans + 1);
}

// lhs block of one (receiver surface, ring surface) pair, one tile per work-group.
template <typename T, int RH, int MODE>  // MODE as SegForm
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 1))) void k_lhs_block(T* __restrict__ lhs, int64_t ld, Receivers<T> rc,
                                                        RingSource<T> src, T sigma, int spans) {
    __shared__ T sv[lhs_stage_values<RH>()];
    lhs_tile<T, RH, MODE>(sv, lhs, ld, rc, src, sigma, blockIdx.x, blockIdx.y, spans);
}

// One (receiver surface, ring surface) block of one influence matrix in a grouped launch: the tiles
// of all sections of all matrices are numbered in section order, section s owning tiles
// [tile0, tile0 + tiles_x tiles_y); tile t of it is receiver block t % tiles_x, ring block t / tiles_x.
template <typename T>
struct LhsSection {
    T* lhs;  // the section's origin in its matrix
    int64_t ld;
    Receivers<T> rc;
    RingSource<T> src;
    int32_t tiles_x, tile0;
    int32_t rh, spans;  // tile shape (lhs_tile_shape)
};

template <typename T>
inline int64_t lhs_tiles_y(const LhsSection<T>& s) {
    const int sw = kWaves * s.spans;
    return (int64_t)((s.src.ns + sw - 1) / sw) * ((s.src.nc + s.rh - 1) / s.rh);
}

// A value every lane of the wave holds alike, moved to a scalar register (the section fields the
// grouped kernel reads from LDS would otherwise sit in vector registers and cost it occupancy).
__device__ __forceinline__ int32_t wave_uniform(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ int64_t wave_uniform(int64_t v) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)((uint64_t)v >> 32));
    return (int64_t)(((uint64_t)hi << 32) | lo);
}
template <typename P>
__device__ __forceinline__ P* wave_uniform(P* p) {
    return reinterpret_cast<P*>(wave_uniform((int64_t)reinterpret_cast<uintptr_t>(p)));
}
template <typename T>
__device__ __forceinline__ LhsSection<T> wave_uniform(const LhsSection<T>& a) {
    LhsSection<T> b;
    b.lhs = wave_uniform(a.lhs);
    b.ld = wave_uniform(a.ld);
    b.rc.colloc = wave_uniform(a.rc.colloc);
    b.rc.cs2 = wave_uniform(a.rc.cs2);
    b.rc.normals = wave_uniform(a.rc.normals);
    b.rc.ns2 = wave_uniform(a.rc.ns2);
    b.rc.m = wave_uniform(a.rc.m);
    b.src.verts = wave_uniform(a.src.verts);
    b.src.vs2 = wave_uniform(a.src.vs2);
    b.src.ns = wave_uniform(a.src.ns);
    b.src.nc = wave_uniform(a.src.nc);
    b.src.wake = wave_uniform(a.src.wake);
    b.src.ws2 = wave_uniform(a.src.ws2);
    b.src.nwv = wave_uniform(a.src.nwv);
    b.src.iteration = wave_uniform(a.src.iteration);
    b.tiles_x = wave_uniform(a.tiles_x);
    b.tile0 = wave_uniform(a.tile0);
    b.rh = wave_uniform(a.rh);
    b.spans = wave_uniform(a.spans);
    return b;
}

// Grouped assembly: many influence matrices of any sizes (different meshes, requests) in one
// launch, one tile per work-group over the work list of all their tiles (the first `tiles`: a
// prefix of whole matrices), numbered section by section; the hardware hands the work-groups out in
// order, so the ones running together work on neighbouring tiles, as in one per-section launch.
// tile0[s] is the first tile of section s (tile0[nsec] = tiles); chunk[c] is the section holding tile
// c * kGroupChunk, so a tile's section is chunk[t / kGroupChunk] or one of the few after it.  Every
// tile runs lhs_tile, so each matrix is bitwise the per-section launches' result.
constexpr int kGroupChunk = 64;

template <typename T, int MODE>
__global__ __launch_bounds__(kThreads) void k_lhs_grouped(const LhsSection<T>* __restrict__ secs,
                                                          const int32_t* __restrict__ tile0,
                                                          const int32_t* __restrict__ chunk, int tiles, T sigma,
                                                          const T* base = nullptr, float* base32 = nullptr) {
    __shared__ T sv[lhs_stage_values<4>()];
    __shared__ LhsSection<T> s_sec;
    const int t = blockIdx.x;
    if (t >= tiles) return;
    if (threadIdx.x == 0) {
        int s = chunk[t / kGroupChunk];
        while (tile0[s + 1] <= t) s++;  // sections are non-empty and tile0 ends with `tiles`
        s_sec = secs[s];
    }
    __syncthreads();
    const LhsSection<T> S = wave_uniform(s_sec);
    const int local = t - S.tile0;
    const int bx = local % S.tiles_x, by = local / S.tiles_x;
    float* l32 = base32 ? base32 + (S.lhs - base) : nullptr;  // with base32 the matrices are set, not added to
    if (S.rh == 4)
        lhs_tile<T, 4, MODE>(sv, S.lhs, S.ld, S.rc, S.src, sigma, bx, by, S.spans, base32 != nullptr, l32);
    else if (S.rh == 2)
        lhs_tile<T, 2, MODE>(sv, S.lhs, S.ld, S.rc, S.src, sigma, bx, by, S.spans, base32 != nullptr, l32);
    else
        lhs_tile<T, 1, MODE>(sv, S.lhs, S.ld, S.rc, S.src, sigma, bx, by, S.spans, base32 != nullptr, l32);
}

// ---- wake influence ---------------------------------------------------------------------------
constexpr int kMaxWakes = TVLM_MAX_SURFACES;

template <typename T>
struct WakeSurface {
    const T* verts;   // {ns+1, nwv, 4} plane contiguous
    int64_t ws2;
    const T* gamma;   // {ns, nwv-1} contiguous
    int32_t ns, nwv;
    int32_t row_begin, row_end;  // ring rows [row_begin, row_end)
    int32_t sw, rh;              // tile extent: spans, rows
    int32_t tiles_span, tile_begin;
    // k_wake_lattice only: a coarse lattice over a finer wake of nsf spans (0: this is the wake
    // itself).  Coarse vertex (column c, row r) is the fine vertex (min(c vcs, nsf), vrow0 + r vrs);
    // coarse ring (r, c) carries the mean circulation of the fine rings of rows
    // [vrow0 + r vrs, vrow0 + (r+1) vrs) and spans [c vcs, min((c+1) vcs, nsf)).
    int32_t vrs = 1, vcs = 1, vrow0 = 0, nsf = 0;
};

template <typename T>
struct WakeTable {
    int32_t n;
    int32_t total_tiles;
    WakeSurface<T> s[kMaxWakes];
};

template <typename T>
struct RecvTable {
    int32_t n;
    int32_t total;
    int32_t offset[kMaxWakes + 1];
    Receivers<T> r[kMaxWakes];
};

constexpr int kTileRings = 256;  // target rings per tile
constexpr int kMaxSpanTile = 64;

template <typename T>
__device__ __forceinline__ int find_surface(const RecvTable<T>& t, int p) {
    int s = 0;
    while (s + 1 < t.n && p >= t.offset[s + 1]) s++;
    return s;
}

// Velocity of the tile's rings with their circulations over one wave's spans [sa, sb), RH rows at a time
// from row q0 on: every segment once with the difference of the circulations beside it (rings outside
// the RH rows, or outside the wave's spans on their far side, add theirs where they are walked).
template <typename T, int RH, int MODE>
__device__ __forceinline__ void wake_walk(const T* sv, const T* sg, int vw, int swe, int rhe, int sa, int sb,
                                          const v3<T>& c, T sigma, v3<T>& acc) {
    using S = SegForm<T, MODE>;
    auto add = [&](const typename S::Seg& s, T g) {
        const T k = g * s.k, km = g * s.km;
        acc.x += k * s.crx + km * s.mrx;
        acc.y += (k - km) * s.cry;
        acc.z += k * s.crz + km * s.mrz;
    };
    typename S::Vertex prev[RH + 1];
#pragma unroll
    for (int q = 0; q <= RH; q++)
        if (q <= rhe) prev[q] = S::vertex(c, sv + 3 * (q * vw + sa));
#pragma unroll 1
    for (int s = sa; s <= sb; s++) {
        // chordwise segments of vertex column s (the tile's right edge with the last span's wave)
        if (s < sb || sb == swe) {
#pragma unroll
            for (int q = 0; q < RH; q++) {
                if (q < rhe) {
                    const T* va = sv + 3 * (q * vw + s);
                    T g = s < swe ? -sg[q * swe + s] : T(0);
                    if (s > 0) g += sg[q * swe + s - 1];
                    add(S::segment(prev[q], prev[q + 1], va, va + 3 * vw, sigma), g);
                }
            }
        }
        if (s == sb) break;
#pragma unroll
        for (int q = 0; q <= RH; q++) {
            if (q <= rhe) {
                const T* va = sv + 3 * (q * vw + s);
                const typename S::Vertex cur = S::vertex(c, va + 3);
                T g = q < rhe ? sg[q * swe + s] : T(0);
                if (q > 0) g -= sg[(q - 1) * swe + s];
                add(S::segment(prev[q], cur, va, va + 3, sigma), g);
                prev[q] = cur;
            }
        }
    }
}

// TS: storage type of the inputs and partials, T: compute type (float for MODE 2).  RH: rows a wave walks
// at a time (the launch's tiles hold more or fewer, wake_tile_shape).  Bound by VALU issue; a call of 400
// receivers x 200 x 40 rings in exact FP64 72.3 -> 44.9 us with the shared segments.
template <typename TS, typename T, int MODE, int RH>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(MODE == 1 ? 1 : 4))) void k_wake_partials(TS* __restrict__ partial, RecvTable<TS> rt,
                                                            WakeTable<TS> wt, T sigma) {
    // LDS: vertex rows of the tile (rh+1) x (sw+1) x 3 and circulations rh x sw.  With
    // rh = floor(kTileRings / sw) and 1 <= sw <= kMaxSpanTile, (rh+1)(sw+1) <= 2 (kTileRings+1).
    __shared__ T sverts[2 * (kTileRings + 1) * 3];
    __shared__ T sgam[kTileRings];
    __shared__ T sred[kWaves][kRecv];

    const int tile = blockIdx.y;
    int w = 0;
    while (w + 1 < wt.n && tile >= wt.s[w + 1].tile_begin) w++;
    const WakeSurface<TS>& ws = wt.s[w];
    const int local = tile - ws.tile_begin;
    const int ts = local % ws.tiles_span, tr = local / ws.tiles_span;
    const int s0 = ts * ws.sw, r0 = ws.row_begin + tr * ws.rh;
    const int swe = min(ws.sw, ws.ns - s0);
    const int rhe = min(ws.rh, ws.row_end - r0);
    const int vw = swe + 1;
    // stage vertex rows r0 .. r0+rhe and circulations
    for (int e = threadIdx.x; e < (rhe + 1) * vw; e += kThreads) {
        const int q = e / vw, sp = e % vw;
        const int64_t g = (int64_t)(s0 + sp) + (int64_t)(r0 + q) * (ws.ns + 1);
        sverts[3 * e + 0] = (T)ws.verts[g];
        sverts[3 * e + 1] = (T)ws.verts[g + ws.ws2];
        sverts[3 * e + 2] = (T)ws.verts[g + 2 * ws.ws2];
    }
    for (int e = threadIdx.x; e < rhe * swe; e += kThreads) {
        const int q = e / swe, sp = e % swe;
        sgam[e] = (T)ws.gamma[(int64_t)(r0 + q) * ws.ns + s0 + sp];
    }
    __syncthreads();

    const int lane = threadIdx.x & (kRecv - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kRecv);
    const int p = blockIdx.x * kRecv + lane;
    const int chunk = (swe + kWaves - 1) / kWaves;
    const int sa = wave * chunk, sb = min(swe, sa + chunk);
    T part = T(0);
    if (p < rt.total && sa < sb) {
        const int si = find_surface(rt, p);
        const Receivers<TS>& rc = rt.r[si];
        const int li = p - rt.offset[si];
        const v3<T> c = {(T)rc.colloc[li], (T)rc.colloc[li + rc.cs2], (T)rc.colloc[li + 2 * rc.cs2]};
        const v3<T> n = {(T)rc.normals[li], (T)rc.normals[li + rc.ns2], (T)rc.normals[li + 2 * rc.ns2]};
        v3<T> acc = {T(0), T(0), T(0)};
#pragma unroll 1
        for (int q0 = 0; q0 < rhe; q0 += RH)
            wake_walk<T, RH, MODE>(sverts + 3 * q0 * vw, sgam + q0 * swe, vw, swe, min(RH, rhe - q0), sa, sb, c, sigma,
                                   acc);
        part = dot(acc, n);
    }
    sred[wave][lane] = part;
    __syncthreads();
    if (wave == 0 && p < rt.total) {
        const T s = (sred[0][lane] + sred[1][lane]) + (sred[2][lane] + sred[3][lane]);
        partial[(int64_t)tile * rt.total + p] = (TS)s;
    }
}

// k_wake_partials with the rows per walk that the launch's tiles hold (the largest of 4, 2, 1 within them).
template <typename T, int MODE>
inline void launch_wake_partials(dim3 grid, hipStream_t st, T* partial, const RecvTable<T>& rt, const WakeTable<T>& wt,
                                 T sigma) {
    int rh = 0;
    for (int m = 0; m < wt.n; m++) rh = wt.s[m].rh > rh ? wt.s[m].rh : rh;
    if (rh >= 4)
        hipLaunchKernelGGL((k_wake_partials<T, T, MODE, 4>), grid, dim3(kThreads), 0, st, partial, rt, wt, sigma);
    else if (rh >= 2)
        hipLaunchKernelGGL((k_wake_partials<T, T, MODE, 2>), grid, dim3(kThreads), 0, st, partial, rt, wt, sigma);
    else
        hipLaunchKernelGGL((k_wake_partials<T, T, MODE, 1>), grid, dim3(kThreads), 0, st, partial, rt, wt, sigma);
}

// rhs[p] -= sum over tiles of partial[tile][p]: 64 receivers per work-group, 16 waves each sum
// every 16th tile, then a fixed-order tree over the waves (bitwise reproducible).
constexpr int kRedWaves = 16;

// sum over t = first, first + step, ... < end of x[t * ld + p], in that order, with the loads of
// eight terms issued before any is added (a plain loop waits for each load in turn).
template <typename T>
__device__ __forceinline__ T strided_sum(const T* __restrict__ x, int64_t ld, int p, int first, int end, int step) {
    T s = T(0);
    for (int t0 = first; t0 < end; t0 += 8 * step) {
        T v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const int t = t0 + k * step;
            v[k] = t < end ? x[(int64_t)t * ld + p] : T(0);
        }
#pragma unroll
        for (int k = 0; k < 8; k++)
            if (t0 + k * step < end) s += v[k];
    }
    return s;
}

template <typename T>
__global__ __launch_bounds__(64 * kRedWaves) void k_wake_reduce(T* __restrict__ rhs, int64_t rhs_stride,
                                                                const T* __restrict__ partial, int tiles, int total) {
    __shared__ T red[kRedWaves][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = blockIdx.x * 64 + lane;
    T s = T(0);
    if (p < total) s = strided_sum(partial, (int64_t)total, p, wave, tiles, kRedWaves);
    red[wave][lane] = s;
    __syncthreads();
#pragma unroll
    for (int h = kRedWaves / 2; h > 0; h >>= 1) {
        if (wave < h) red[wave][lane] += red[wave + h][lane];
        __syncthreads();
    }
    if (wave == 0 && p < total) rhs[(int64_t)p * rhs_stride] -= red[0][lane];
}

template <typename T>
inline void launch_wake_reduce(T* rhs, int64_t rhs_stride, const T* partial, int tiles, int total, hipStream_t st) {
    hipLaunchKernelGGL(k_wake_reduce<T>, dim3((total + 63) / 64), dim3(64 * kRedWaves), 0, st, rhs, rhs_stride, partial,
                       tiles, total);
}

// Tile shape of one wake surface: spans per tile sw <= kMaxSpanTile, rows per tile rh with
// rh * sw <= kTileRings, as few rows as keep the launch within wake_target_groups() work-groups
// (receiver blocks x tiles).  A tile's rows share the segments between them, so that two rows are taken for one
// where that leaves a fifth of the target: 400 receivers x 40 spans, 200 rows: 45 us with two rows (700 work-groups),
// 52 with one; 100 rows: 34 (350) and 31; 85 receivers x 17 spans x 500 rows: 23 (500) and 25.  Three rows are walked
// as two and one, and four took 194 us where they took 229 (1800 receivers x 60 spans x 200 rows).
inline void wake_tile_shape(int ns, int rows, int recv_blocks, int& sw, int& rh) {
    sw = ns < kMaxSpanTile ? ns : kMaxSpanTile;
    const int tiles_span = (ns + sw - 1) / sw;
    const int64_t groups = (int64_t)recv_blocks * tiles_span;  // per row tile
    int rh_max = kTileRings / sw;
    if (rh_max < 1) rh_max = 1;
    int64_t want_row_tiles = wake_target_groups() / groups;
    if (want_row_tiles < 1) want_row_tiles = 1;
    rh = (int)((rows + want_row_tiles - 1) / want_row_tiles);
    if (rh <= 1) rh = (rows + 1) / 2 * groups * 5 >= wake_target_groups() ? 2 : 1;
    if (rh == 3) rh = 4;
    if (rh > rh_max) rh = rh_max;
}

// Wake induction of the seeded FP64 form evaluated on the vortex lattice.  Every segment of the
// tile is evaluated once with strength = difference of the circulations of the two rings that share
// it (spanwise segment of vertex row q, span s: G(q,s) - G(q-1,s); chordwise segment of vertex
// column s: G(q,s-1) - G(q,s); rings outside the work-group tile count 0 -- their own tile adds
// them).  The work-group tile is RH rows x up to 4*CH spans; wave w walks the ring columns of its
// span chunk left to right keeping the vertex terms of the previous vertex column in registers, so
// a ring costs (RH+1)/RH vertex terms and (2 RH + 1)/RH segments (both images share x and z).
struct LatVertex {
    double x, y, z, ri;  // c - v, 1/|c - v|
    double ym, rim;      // image receiver (y -> -y): y component and 1/|.|
};

__device__ __forceinline__ LatVertex lat_vertex(double cx, double cy, double cz, const double* v) {
    LatVertex f;
    f.x = cx - v[0];
    f.y = cy - v[1];
    f.z = cz - v[2];
    f.ym = -cy - v[1];
    const double xz = f.x * f.x + f.z * f.z;
    f.ri = rsqrt_seeded(xz + f.y * f.y);
    f.rim = rsqrt_seeded(xz + f.ym * f.ym);
    return f;
}

constexpr int kLatChunkMax = 16;  // spans per wave

// A segment a -> b of a staged tile: b - a, and the difference of the circulations beside it.
struct LatSegment {
    double x, y, z, g;
};

// What a work-group stages of a tile of RH rings x 4 kLatChunkMax spans.
template <int RH>
struct LatTile {
    static constexpr int kSpans = kWaves * kLatChunkMax;
    double verts[(RH + 1) * (kSpans + 1) * 3];  // vertex rows 0..rhe x vw = swe + 1 columns
    double gam[RH * kSpans];                    // circulations rhe x swe
    LatSegment span[(RH + 1) * kSpans];         // vertex row q, from vertex column s to s + 1: q * swe + s
    LatSegment chord[RH * (kSpans + 1)];        // vertex column s, from vertex row q to q + 1: q * vw + s
    int small;                                  // not 0: some ring is so small that its segments meet the cutoffs
};

// The segments of a tile whose vertices and circulations are staged (between two barriers).  Rings
// outside the tile count 0 in the differences: their own tile adds them.  A receiver in line with a ring's
// middle has |r1 x r2| of half the ring's area with its chordwise edges, wherever along the line it stands: rings
// whose half is below the cutoff, within a tenth, set t.small (0 before).
template <int RH>
__device__ __forceinline__ void lattice_segments(LatTile<RH>& t, int swe, int rhe) {
    const int vw = swe + 1;
    for (int e = threadIdx.x; e < (rhe + 1) * swe; e += kThreads) {
        const int q = e / swe, s = e % swe;
        const double* v = t.verts + 3 * (q * vw + s);
        double g = 0.0;
        if (q < rhe) g += t.gam[q * swe + s];
        if (q > 0) g -= t.gam[(q - 1) * swe + s];
        t.span[e] = {v[3] - v[0], v[4] - v[1], v[5] - v[2], g};
    }
    for (int e = threadIdx.x; e < rhe * vw; e += kThreads) {
        const int q = e / vw, s = e % vw;
        const double *v = t.verts + 3 * e, *w = v + 3 * vw;
        double g = 0.0;
        if (s < swe) g -= t.gam[q * swe + s];
        if (s > 0) g += t.gam[q * swe + s - 1];
        const double x = w[0] - v[0], y = w[1] - v[1], z = w[2] - v[2];
        t.chord[e] = {x, y, z, g};
        if (s < swe) {
            const double sx = v[3] - v[0], sy = v[4] - v[1], sz = v[5] - v[2];
            const double nx = y * sz - z * sy, ny = z * sx - x * sz, nz = x * sy - y * sx;
            if (nx * nx + ny * ny + nz * nz < 4.4 * BS<double>::cut_cross) t.small = 1;
        }
    }
}

__device__ __forceinline__ uint32_t hi_word(double v) { return (uint32_t)__double2hiint(v); }

// A staged segment a->b for the receiver and for its image in y = 0, without the 1/(4 pi) factor (lattice_chunk
// applies it once to its sum).  The two share every term without a y component: the y component of r1 x r2
// and its square, and the x and z parts of r0.r1 and r0.r2.
__device__ __forceinline__ void lat_pair(double& ax, double& ay, double& az, const LatVertex& a, const LatVertex& b,
                                         const LatSegment& r) {
    const double cry = a.z * b.x - a.x * b.z;
    const double cry2 = cry * cry;
    const double d1xz = r.x * a.x + r.z * a.z;
    const double d2xz = r.x * b.x + r.z * b.z;
    constexpr double cut = BS<double>::cut_cross;
    // |r| < RCUT  <=>  1/|r| > 1/RCUT
    constexpr double rimax = 1.0 / BS<double>::cut_norm;
    {
        const double crx = a.y * b.z - a.z * b.y;
        const double crz = a.x * b.y - a.y * b.x;
        const double sq = crx * crx + crz * crz + cry2;
        const double d1 = d1xz + r.y * a.y, d2 = d2xz + r.y * b.y;
        const bool ok = (sq >= cut) & (a.ri <= rimax) & (b.ri <= rimax);
        const double t = (d1 * a.ri - d2 * b.ri) * rcp_seeded(sq) * r.g;
        const double coeff = ok ? t : 0.0;
        ax += coeff * crx;
        ay += coeff * cry;
        az += coeff * crz;
    }
    {
        const double crx = a.ym * b.z - a.z * b.ym;
        const double crz = a.x * b.ym - a.ym * b.x;
        const double sq = crx * crx + crz * crz + cry2;
        const double d1 = d1xz + r.y * a.ym, d2 = d2xz + r.y * b.ym;
        const bool ok = (sq >= cut) & (a.rim <= rimax) & (b.rim <= rimax);
        const double t = (d1 * a.rim - d2 * b.rim) * rcp_seeded(sq) * r.g;
        const double coeff = ok ? t : 0.0;
        ax += coeff * crx;
        ay -= coeff * cry;
        az += coeff * crz;
    }
}

// A staged segment for the receiver and its image, as lat_pair but without its cutoffs: low_sq keeps
// the smallest high word of |r1 x r2|^2 met, so that the walk learns at its end whether any segment came
// near a cutoff.  The image shares every term without a y component and the one reciprocal,
// 1/(sq sq') = the seeded estimate, of which each takes its part: 46 issue slots (of one FP64
// multiply-add) a pair of segments, where lat_pair with its compares and selects takes 58.
__device__ __forceinline__ void lat_pair_fast(double& ax, double& ay, double& az, const LatVertex& a,
                                              const LatVertex& b, const LatSegment& r, uint32_t& low_sq) {
    const double cry = a.z * b.x - a.x * b.z;
    const double cry2 = cry * cry;
    const double d1xz = r.x * a.x + r.z * a.z;
    const double d2xz = r.x * b.x + r.z * b.z;
    const double crx = a.y * b.z - a.z * b.y, crz = a.x * b.y - a.y * b.x;
    const double mrx = a.ym * b.z - a.z * b.ym, mrz = a.x * b.ym - a.ym * b.x;
    const double sq = crx * crx + (crz * crz + cry2), sqm = mrx * mrx + (mrz * mrz + cry2);
    const double inv = rcp_seeded(sq * sqm) * r.g;
    const double t = ((d1xz + r.y * a.y) * a.ri - (d2xz + r.y * b.y) * b.ri) * (inv * sqm);
    const double tm = ((d1xz + r.y * a.ym) * a.rim - (d2xz + r.y * b.ym) * b.rim) * (inv * sq);
    low_sq = min(min(low_sq, hi_word(sq)), hi_word(sqm));
    ax += t * crx;
    ay += t * cry;
    az += t * crz;
    ax += tm * mrx;
    ay -= tm * cry;
    az += tm * mrz;
}

// lat_vertex, with the smallest high word of |r|^2 kept in low_r2.
__device__ __forceinline__ LatVertex lat_vertex_fast(double cx, double cy, double cz, const double* v,
                                                     uint32_t& low_r2) {
    LatVertex f;
    f.x = cx - v[0];
    f.y = cy - v[1];
    f.z = cz - v[2];
    f.ym = -cy - v[1];
    const double xz = f.x * f.x + f.z * f.z;
    const double r2 = xz + f.y * f.y, r2m = xz + f.ym * f.ym;
    f.ri = rsqrt_seeded(r2);
    f.rim = rsqrt_seeded(r2m);
    low_r2 = min(min(low_r2, hi_word(r2)), hi_word(r2m));
    return f;
}

// The lattice walk of one wave over its span chunk [sa, sb) of a staged tile for the receiver
// (cx, cy, cz): chordwise segments of each vertex column, spanwise segments of each vertex row, the
// previous vertex column's terms kept in registers; the tile's right edge only when sb == swe.  (ax, ay, az): 4 pi x
// the induced velocity.  CUT: every cutoff is applied where it stands; else none is, and low_sq and low_r2 are
// the smallest high words of |r1 x r2|^2 and |r|^2 met.
template <int RH, bool CUT>
__device__ __forceinline__ void lattice_walk(const LatTile<RH>& t, int swe, int rhe, int sa, int sb, double cx, double cy,
                                             double cz, double& ax, double& ay, double& az, uint32_t& low_sq,
                                             uint32_t& low_r2) {
    const int vw = swe + 1;
    auto vertex = [&](int q, int s) {
        const double* v = t.verts + 3 * (q * vw + s);
        if constexpr (CUT)
            return lat_vertex(cx, cy, cz, v);
        else
            return lat_vertex_fast(cx, cy, cz, v, low_r2);
    };
    auto pair = [&](const LatVertex& a, const LatVertex& b, const LatSegment& r) {
        if constexpr (CUT)
            lat_pair(ax, ay, az, a, b, r);
        else
            lat_pair_fast(ax, ay, az, a, b, r, low_sq);
    };
    ax = ay = az = 0.0;
    LatVertex prev[RH + 1];
#pragma unroll
    for (int q = 0; q <= RH; q++)
        if (q <= rhe) prev[q] = vertex(q, sa);
    for (int s = sa; s < sb; s++) {
        // chordwise segments of vertex column s (left edge of ring column s)
#pragma unroll
        for (int q = 0; q < RH; q++)
            if (q < rhe) pair(prev[q], prev[q + 1], t.chord[q * vw + s]);
        // vertex column s+1 and the spanwise segments of ring column s
#pragma unroll
        for (int q = 0; q <= RH; q++) {
            if (q <= rhe) {
                const LatVertex cur = vertex(q, s + 1);
                pair(prev[q], cur, t.span[q * swe + s]);
                prev[q] = cur;
            }
        }
    }
    if (sb == swe) {  // right edge of the work-group tile: chordwise segments of vertex column swe
#pragma unroll
        for (int q = 0; q < RH; q++)
            if (q < rhe) pair(prev[q], prev[q + 1], t.chord[q * vw + swe]);
    }
}

// A wave's walk without the cutoffs, taken again with them where some lane's smallest |r1 x r2|^2 or |r|^2 is
// within a rounding of its cutoff or below it, or a result is not finite (an input that is not, or a
// product that overflowed); tiles of rings so small that this is to be expected (t.small) are walked with
// them from the start.  Adds the induced velocity to (vx, vy, vz).
// Bound by FP64 VALU issue.  Per (receiver, ring) pair at RH = 4: 2.25 segment pairs of 46 slots and
// 1.25 vertices of 25 against 58 and 24 with the cutoffs inside.  The cutoffs are absolute (1e-10): a 10 x 40 wing of
// chord 1 hardly meets them, one of chord 0.05 or less in nearly every tile beside it.
// 300 steps of 16 such simulations at chord 1, 0.1, 0.05 and 0.01: 68.3, 68.7, 78.1 and 78.7 ms; with the cutoffs
// inside throughout 81 to 82, with none inside and t.small not tested 67.9, 68.6, 102 and 166.
template <int RH>
__device__ __forceinline__ void lattice_chunk(const LatTile<RH>& t, int swe, int rhe, int sa, int sb, double cx,
                                              double cy, double cz, double& vx, double& vy, double& vz) {
    double ax = 0.0, ay = 0.0, az = 0.0;
    uint32_t low_sq = 0xffffffffu, low_r2 = 0xffffffffu;
    bool careful = __builtin_amdgcn_readfirstlane(t.small) != 0;
    if (!careful) {
        lattice_walk<RH, false>(t, swe, rhe, sa, sb, cx, cy, cz, ax, ay, az, low_sq, low_r2);
        constexpr double cut_r2 = BS<double>::cut_norm * BS<double>::cut_norm;
        const bool near = (low_sq <= hi_word(BS<double>::cut_cross)) | (low_r2 <= hi_word(cut_r2)) |
                          !(fabs(ax) + fabs(ay) + fabs(az) < __builtin_huge_val());
        careful = __ballot(near) != 0ull;
    }
    if (careful) lattice_walk<RH, true>(t, swe, rhe, sa, sb, cx, cy, cz, ax, ay, az, low_sq, low_r2);
    constexpr double inv_fourpi = 1.0 / BS<double>::fourpi;
    vx += ax * inv_fourpi;
    vy += ay * inv_fourpi;
    vz += az * inv_fourpi;
}

// zs: simulations (blockIdx.z) of one launch find their receivers, wake and circulations z * zs
// elements after simulation 0's (the tables' pointers) and write their partials z * wzs after.
// At least 4 waves per SIMD (the hint keeps a later change from dropping a wave unnoticed).
template <typename TS, int RH>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4))) void k_wake_lattice(TS* __restrict__ partial, RecvTable<TS> rt,
                                                           WakeTable<TS> wt, int64_t zs = 0, int64_t wzs = 0) {
    const int64_t zo = (int64_t)blockIdx.z * zs;
    partial += (int64_t)blockIdx.z * wzs;
    __shared__ LatTile<RH> st;
    if (threadIdx.x == 0) st.small = 0;
    double *const sverts = st.verts, *const sgam = st.gam;
    __shared__ double sred[kWaves][kRecv];
    const int tile = blockIdx.y;
    int w = 0;
    while (w + 1 < wt.n && tile >= wt.s[w + 1].tile_begin) w++;
    const WakeSurface<TS>& ws = wt.s[w];
    const int local = tile - ws.tile_begin;
    const int ts = local % ws.tiles_span, tr = local / ws.tiles_span;
    const int s0 = ts * ws.sw, r0 = ws.row_begin + tr * ws.rh;
    const int swe = min(ws.sw, ws.ns - s0);
    const int rhe = min(ws.rh, ws.row_end - r0);
    const int vw = swe + 1;
    const int nsf = ws.nsf ? ws.nsf : ws.ns;
    for (int e = threadIdx.x; e < (rhe + 1) * vw; e += kThreads) {
        const int q = e / vw, sp = e % vw;
        const int col = min((s0 + sp) * ws.vcs, nsf);
        const int64_t g = zo + (int64_t)col + (int64_t)(ws.vrow0 + (r0 + q) * ws.vrs) * (nsf + 1);
        sverts[3 * e + 0] = (double)ws.verts[g];
        sverts[3 * e + 1] = (double)ws.verts[g + ws.ws2];
        sverts[3 * e + 2] = (double)ws.verts[g + 2 * ws.ws2];
    }
    if (ws.vrs == 1 && ws.vcs == 1) {
        for (int e = threadIdx.x; e < rhe * swe; e += kThreads) {
            const int q = e / swe, sp = e % swe;
            sgam[e] = (double)ws.gamma[zo + (int64_t)(ws.vrow0 + r0 + q) * nsf + s0 + sp];
        }
    } else {  // coarse ring: mean of the fine rings it replaces, rows then spans in order
        for (int e = threadIdx.x; e < rhe * swe; e += kThreads) {
            const int q = e / swe, sp = e % swe;
            const int fr0 = ws.vrow0 + (r0 + q) * ws.vrs, fc0 = (s0 + sp) * ws.vcs;
            const int fc1 = min(fc0 + ws.vcs, nsf);
            double sum = 0.0;
            for (int fr = fr0; fr < fr0 + ws.vrs; fr++)
                for (int fc = fc0; fc < fc1; fc++) sum += (double)ws.gamma[zo + (int64_t)fr * nsf + fc];
            sgam[e] = sum / (double)(ws.vrs * (fc1 - fc0));
        }
    }
    __syncthreads();
    lattice_segments<RH>(st, swe, rhe);
    __syncthreads();
    const int lane = threadIdx.x & (kRecv - 1);
    const int wave = threadIdx.x / kRecv;
    const int p = blockIdx.x * kRecv + lane;
    double part = 0.0;
    const int chunk = (swe + kWaves - 1) / kWaves;
    const int sa = wave * chunk, sb = min(swe, sa + chunk);
    if (p < rt.total && sa < sb) {
        const int si = find_surface(rt, p);
        const Receivers<TS>& rc = rt.r[si];
        const int li = p - rt.offset[si];
        const TS* co = rc.colloc + zo;
        const TS* no = rc.normals + zo;
        const double cx = co[li], cy = co[li + rc.cs2], cz = co[li + 2 * rc.cs2];
        double ax = 0.0, ay = 0.0, az = 0.0;
        lattice_chunk<RH>(st, swe, rhe, sa, sb, cx, cy, cz, ax, ay, az);
        part = ax * (double)no[li] + ay * (double)no[li + rc.ns2] + az * (double)no[li + 2 * rc.ns2];
    }
    sred[wave][lane] = part;
    __syncthreads();
    if (wave == 0 && p < rt.total)
        partial[(int64_t)tile * rt.total + p] = (TS)((sred[0][lane] + sred[1][lane]) + (sred[2][lane] + sred[3][lane]));
}

// Tile shape for k_wake_lattice: sw <= 4 * kLatChunkMax spans, rh in {1, 2, 4} rows, chosen so
// that the launch has about kLatTargetGroups work-groups.

inline void lattice_tile_shape(int ns, int rows, int recv_blocks, int& sw, int& rh) {
    sw = ns < kWaves * kLatChunkMax ? ns : kWaves * kLatChunkMax;
    const int tiles_span = (ns + sw - 1) / sw;
    int want_row_tiles = kLatTargetGroups / (recv_blocks * tiles_span);
    if (want_row_tiles < 1) want_row_tiles = 1;
    const int need = (rows + want_row_tiles - 1) / want_row_tiles;
    rh = need <= 1 ? 1 : need <= 2 ? 2 : 4;
}

// Span extent of a lattice tile when the launch's spans are split `split` ways: ceil(ns / split)
// spans, at least 2 per wave (or all ns), at most kWaves * kLatChunkMax.
inline int lattice_span_tile(int ns, int split) {
    int sw = (ns + split - 1) / split;
    const int lo = ns < 2 * kWaves ? ns : 2 * kWaves;
    if (sw < lo) sw = lo;
    if (sw > kWaves * kLatChunkMax) sw = kWaves * kLatChunkMax;
    return sw;
}

// One shape for every surface of a k_wake_lattice launch (rows per tile rh, the kernel's template
// value, and a span split): a launch of more than `target` work-groups with one row per tile takes
// 2 or 4 rows per tile (the smallest that gets within the target, else 4); a smaller launch splits
// its spans (2, 3, ... ways, at least 2 spans per wave) until it reaches the target or cannot split
// further, so that a short wake still spreads over the CUs.  A split launch holds fewer than
// 2 target work-groups.
template <typename T>
inline void lattice_launch_shape(const WakeTable<T>& wt, int recv_blocks, int target, int& rh, int& split) {
    auto groups = [&](int rh_, int k) {
        int64_t g = 0;
        for (int m = 0; m < wt.n; m++) {
            const WakeSurface<T>& w = wt.s[m];
            const int sw = lattice_span_tile(w.ns, k);
            g += (int64_t)recv_blocks * ((w.ns + sw - 1) / sw) * ((w.row_end - w.row_begin + rh_ - 1) / rh_);
        }
        return g;
    };
    rh = 1;
    split = 1;
    if (groups(1, 1) > target) {
        rh = groups(2, 1) <= target ? 2 : 4;
        return;
    }
    for (int k = 2; k <= 64 && groups(1, split) < target; k++) {
        bool finer = false;  // does k split any surface finer than the current split?
        for (int m = 0; m < wt.n; m++)
            if (lattice_span_tile(wt.s[m].ns, k) < lattice_span_tile(wt.s[m].ns, split)) finer = true;
        if (!finer) continue;
        if (groups(1, k) > 2 * (int64_t)target) break;
        split = k;
    }
}

}  // namespace
}  // namespace tvlm
