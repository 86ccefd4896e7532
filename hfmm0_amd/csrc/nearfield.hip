// Near field (P2P) of the FMM for gfx950: FP64 and mixed-precision potentials, and the potential
// with the field E = -grad phi.
//
// A work item (NearItem) is a chunk of up to 64 R targets of one leaf; a workgroup of kNearWaves
// waves takes it.  Each lane holds R targets of the chunk (li, li + L, ..., with L lanes per group,
// L = next power of two >= chunk / R) and scans every G-th source (G = 64 / L groups) of 64-source
// batches staged in LDS, so that every source read from LDS feeds R independent pair evaluations.
// The waves take the leaf's batches in turn (wave w batches w, w + kNearWaves, ...), each with its
// own stage, so no wave waits for another before their sums meet in LDS.  The host splits a leaf
// into more, smaller chunks where its pairs would outlast the rest of the launch, and orders the
// items longest first (plan.cpp, near_items).
//
// A leaf's sources are ranges of consecutive points.  Per batch, a record holds the range of its
// first source and a mask of the sources at which a new range starts, so that a lane finds its
// point with a population count and one load instead of a walk along the ranges; the record, that
// load and the points of the next batches are fetched while the current one is evaluated.
//
// Bound by the issue of the pair arithmetic where the leaves are many and alike: 520 G pairs/s in
// FP64 (400k points in a cube, 9.3e8 pairs, 1.78 ms), 1.2 T pairs/s mixed (1M, 7.7e8, 0.64 ms).
// Against one wave per leaf that walked the ranges (same arithmetic), where the latencies of the
// heaviest leaf were the kernel's time: 640 points 23.4 -> 5.0 us, 400k FP64 2.65 -> 1.78 ms, 40k with the
// field (one leaf 38 times the mean) 0.47 -> 0.085 ms, 60k on surfaces FP64 0.52 -> 0.12 ms; mixed:
// 100k 1.09 -> 0.16 ms, 300k on surfaces 2.64 -> 0.46 ms, 150k at k = 0 0.144 -> 0.090 ms, 1M 0.665 ->
// 0.642 ms; 16 problems of 2k to 20k in FP64 0.98 -> 0.27 ms.
#include <hip/hip_runtime.h>

#include <string>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "p2p_math.h"

namespace hfmm {

namespace {

using nearfield::HalfTurnK;
using nearfield::SinCosPi64;

constexpr int kNearThreads = 64 * kNearWaves;

// e^{ikr}/r and the field weight (1 - ikr) e^{ikr}/r^3, so that
// -grad_x e^{ik|x-y|}/|x-y| = (x - y) * field weight (HFMM.py:29-37 in complex form)
__device__ inline void field_weights(float r2, float k, float& wr, float& wi, float& fr, float& fi) {
    nearfield::radian_weight(r2, k, wr, wi);
    const float rinv2 = 1.0f / r2;
    const float kr = k * sqrtf(r2);
    fr = (wr + kr * wi) * rinv2;
    fi = (wi - kr * wr) * rinv2;
}
__device__ inline void field_weights64(double r2, double fl2, double k, HalfTurnK kp, const SinCosPi64& sp, double& wr,
                                       double& wi, double& fr, double& fi) {
    double c, s, rs, rinv, r;
    nearfield::halfturn64(r2, kp, sp, c, s, rs, rinv, r);
    rs = r2 > fl2 ? rs : 0.0;
    wr = c * rs;
    wi = s * rs;
    const double kr = k * r, rinv2 = rs * rs;
    fr = fma(kr, wi, wr) * rinv2;
    fi = fma(-kr, wr, wi) * rinv2;
}

// The forms of the pair arithmetic.  A form has the doubles of LDS its stage takes (kStage, 64
// sources), the real sums per target (kSums), the type of the sums within a batch (Acc; added into
// FP64 sums after each), a target's position (Pos), and
//   pos(x, y, z)             of a point relative to the leaf centre,
//   stage(st, lane, ...)     a source (relative position, charge) into the stage,
//   load(st, j)              a staged source (Src),
//   pair(t, src, acc)        one pair into the sums,
//   apart(t, src)            (kSkips) r^2 above the floor: pairs at it enter with the weight zero, which
//                            is nothing where the charge is finite; else they are left out.

template <typename Pos, typename Src>
__device__ __forceinline__ bool apart_at(const Pos& t, const Src& s, double fl2) {
    const double dx = t.x - s.x, dy = t.y - s.y, dz = t.z - s.z;
    return dx * dx + dy * dy + dz * dz > fl2;
}

// FP64 throughout.  Pairs at or below the leaf's coincidence floor get the weight zero.  About 50
// FP64 instructions a pair with a v_rsq_f64 (45 FP64 of 58 VALU): 9.3e8 pairs took 2.65 ms in a kernel
// of one wave per leaf, where the device library's sincos, square root and division took 5.41; 1.77 ms
// over work items.
struct FormFp64 {
    static constexpr int kStage = 5 * 64, kSums = 2;
    static constexpr bool kSkips = true;
    using Acc = double;
    struct Pos { double x, y, z; };
    struct Src { double x, y, z, qr, qi; };
    double fl2;
    HalfTurnK kp;
    SinCosPi64 sp;
    __device__ FormFp64(const P2PArgs& a, int leaf)
        : fl2(a.floor2[leaf]), kp{a.kp_hi, a.kp_lo}, sp(SinCosPi64::pinned()) {}
    __device__ Pos pos(double x, double y, double z) const { return {x, y, z}; }
    __device__ void stage(double* st, int lane, double x, double y, double z, double2 q) const {
        st[lane] = x;
        st[64 + lane] = y;
        st[128 + lane] = z;
        st[192 + lane] = q.x;
        st[256 + lane] = q.y;
    }
    __device__ Src load(const double* st, int j) const { return {st[j], st[64 + j], st[128 + j], st[192 + j], st[256 + j]}; }
    __device__ bool apart(const Pos& t, const Src& s) const { return apart_at(t, s, fl2); }
    __device__ void pair(const Pos& t, const Src& s, double* acc) const {
        const double dx = t.x - s.x, dy = t.y - s.y, dz = t.z - s.z;
        const double r2 = dx * dx + dy * dy + dz * dz;
        double wr, wi;
        nearfield::pair_weight64(r2, fl2, kp, sp, wr, wi);
        acc[0] = fma(wr, s.qr, fma(-wi, s.qi, acc[0]));
        acc[1] = fma(wr, s.qi, fma(wi, s.qr, acc[1]));
    }
};

__device__ __forceinline__ void add_pair32(float wr, float wi, float2 q, float* acc) {
    acc[0] = fmaf(wr, q.x, acc[0]);
    acc[0] = fmaf(-wi, q.y, acc[0]);
    acc[1] = fmaf(wr, q.y, acc[1]);
    acc[1] = fmaf(wi, q.x, acc[1]);
}

// Mixed precision: coordinates relative to the target leaf centre and scaled by a.scale = k / pi,
// coordinate differences and r^2 in FP64 (exact to rounding for close pairs), weights
// e^{i pi u}/u (u = k r / pi) in FP32 (PH: phase in FP64), the sums of a batch in FP32.  LOWK
// (k r below 1e-4 over every pair of the plan, k = 0 included): coordinates unscaled and the
// weights 1/r + i k, exact to FP32 rounding.  The floor is at least 2^-120, so that an FP32 r^2
// above it is a normal number.
template <bool PH, bool LOWK>
struct FormMixed {
    static constexpr int kStage = 4 * 64, kSums = 2;
    static constexpr bool kSkips = false;
    using Acc = float;
    struct Pos { double x, y, z; };
    struct Src { double x, y, z; float2 q; };
    double sc, fl2;
    float kf;
    __device__ FormMixed(const P2PArgs& a, int leaf)
        : sc(a.scale), fl2(fmax(a.floor2[leaf] * a.scale * a.scale, 0x1p-120)), kf((float)a.k) {}
    __device__ Pos pos(double x, double y, double z) const { return {x * sc, y * sc, z * sc}; }
    __device__ void stage(double* st, int lane, double x, double y, double z, double2 q) const {
        const float2 qf = make_float2((float)q.x, (float)q.y);
        ((double2*)st)[lane] = make_double2(x * sc, y * sc);
        ((double2*)st)[64 + lane] = make_double2(z * sc, __builtin_bit_cast(double, qf));
    }
    __device__ Src load(const double* st, int j) const {
        const double2 xy = ((const double2*)st)[j], zq = ((const double2*)st)[64 + j];
        return {xy.x, xy.y, zq.x, __builtin_bit_cast(float2, zq.y)};
    }
    __device__ void pair(const Pos& t, const Src& s, float* acc) const {
        const double dx = t.x - s.x, dy = t.y - s.y, dz = t.z - s.z;
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        float wr, wi;
        if constexpr (LOWK) {
            const bool ok = r2 > fl2;
            const float rs = nearfield::rsq((float)r2);
            wr = ok ? rs : 0.0f;
            wi = ok ? kf : 0.0f;
        } else {
            nearfield::pair_weight<PH>(r2, fl2, wr, wi);
        }
        add_pair32(wr, wi, s.q, acc);
    }
};

// Mixed precision with the scaled coordinates rounded to FP32 once, coordinate differences and r^2
// in FP32: the FP32-phase leaves flagged in a.coord32
struct FormMixed32 {
    static constexpr int kStage = 4 * 64, kSums = 2;
    static constexpr bool kSkips = false;
    using Acc = float;
    struct Pos { float x, y, z; };
    struct Src { float4 p; float2 q; };
    double sc;
    float fl2;
    __device__ FormMixed32(const P2PArgs& a, int leaf)
        : sc(a.scale), fl2((float)fmax(a.floor2[leaf] * a.scale * a.scale, 0x1p-120)) {}
    __device__ Pos pos(double x, double y, double z) const { return {(float)(x * sc), (float)(y * sc), (float)(z * sc)}; }
    __device__ void stage(double* st, int lane, double x, double y, double z, double2 q) const {
        ((float4*)st)[lane] = make_float4((float)(x * sc), (float)(y * sc), (float)(z * sc), 0.0f);
        ((float2*)(st + 128))[lane] = make_float2((float)q.x, (float)q.y);
    }
    __device__ Src load(const double* st, int j) const { return {((const float4*)st)[j], ((const float2*)(st + 128))[j]}; }
    __device__ void pair(const Pos& t, const Src& src, float* acc) const {
        const float dx = t.x - src.p.x, dy = t.y - src.p.y, dz = t.z - src.p.z;
        const float r2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
        float c, s, rs;
        nearfield::halfturn_parts(fmaxf(r2, 0x1p-120f), c, s, rs);
        rs = r2 > fl2 ? rs : 0.0f;
        add_pair32(c * rs, s * rs, src.q, acc);
    }
};

// The potential and the field, in T.  Coordinates relative to the leaf centre and r^2 in FP64 at
// every precision: FP32 coordinates would carry an absolute error of 2^-24 times the leaf size, a
// large relative error of r for close pairs (points on surfaces); FP64 adds and FMAs issue at the
// rate of the (unpacked) FP32 ones.
template <typename T, bool PH>
struct FormField {
    static constexpr int kStage = 5 * 64, kSums = 8;   // phi, Ex, Ey, Ez (re, im)
    static constexpr bool kSkips = std::is_same<T, double>::value;
    using Acc = T;
    struct Pos { double x, y, z; };
    struct Src { double x, y, z; T qr, qi; };
    double fl2, k;
    T kk;
    HalfTurnK kp;
    SinCosPi64 sp;
    __device__ FormField(const P2PArgs& a, int leaf)
        : fl2(a.floor2[leaf]), k(a.k), kk((T)a.k), kp{a.kp_hi, a.kp_lo}, sp(SinCosPi64::pinned()) {}
    __device__ Pos pos(double x, double y, double z) const { return {x, y, z}; }
    __device__ void stage(double* st, int lane, double x, double y, double z, double2 q) const {
        st[lane] = x;
        st[64 + lane] = y;
        st[128 + lane] = z;
        ((T*)(st + 192))[lane] = (T)q.x;
        ((T*)(st + 256))[lane] = (T)q.y;
    }
    __device__ Src load(const double* st, int j) const {
        return {st[j], st[64 + j], st[128 + j], ((const T*)(st + 192))[j], ((const T*)(st + 256))[j]};
    }
    __device__ bool apart(const Pos& t, const Src& s) const { return apart_at(t, s, fl2); }
    __device__ void pair(const Pos& t, const Src& s, T* acc) const {
        const double dx = t.x - s.x, dy = t.y - s.y, dz = t.z - s.z;
        const double r2 = dx * dx + dy * dy + dz * dz;
        if (!std::is_same<T, double>::value && !(r2 > fl2)) return;   // FP64: zero weights at the floor
        T wr, wi, fr, fi;
        if constexpr (std::is_same<T, double>::value) {
            field_weights64(r2, fl2, k, kp, sp, wr, wi, fr, fi);
        } else if constexpr (PH) {
            float rinv, kr;
            nearfield::radian_weight_phase64(r2, k, wr, wi, rinv, kr);
            const float rinv2 = rinv * rinv;
            fr = (wr + kr * wi) * rinv2;
            fi = (wi - kr * wr) * rinv2;
        } else {
            field_weights((T)r2, kk, wr, wi, fr, fi);
        }
        acc[0] += wr * s.qr - wi * s.qi;
        acc[1] += wr * s.qi + wi * s.qr;
        const T gr = fr * s.qr - fi * s.qi, gi = fr * s.qi + fi * s.qr;
        acc[2] += (T)dx * gr;
        acc[3] += (T)dx * gi;
        acc[4] += (T)dy * gr;
        acc[5] += (T)dy * gi;
        acc[6] += (T)dz * gr;
        acc[7] += (T)dz * gi;
    }
};

// conjugate for k < 0 (the kernels compute with |k|); real for k == 0 with real charges
__device__ __forceinline__ double2 out_value(double2 f, int out_mode) {
    if (out_mode & 1) f.y = -f.y;
    if (out_mode & 2) f.y = 0.0;
    return f;
}

template <class F, int R>
constexpr int near_lds_doubles() {
    return kNearWaves * (F::kStage > 64 * R * F::kSums ? F::kStage : 64 * R * F::kSums);
}

// One work item.  The target sums (times a.wscale, k / pi for the scaled mixed forms) are added to
// the far field and written in input order.
template <class F, int R>
__device__ __forceinline__ void near_body(const P2PArgs& a, const NearItem item, double* lds) {
    constexpr int NS = F::kSums;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int leaf = item.leaf, tc = item.n_targets;
    const F f(a, leaf);
    const double cx = a.bx.centre[3 * item.box], cy = a.bx.centre[3 * item.box + 1], cz = a.bx.centre[3 * item.box + 2];
    const int S = a.leaf_src_total[leaf], n_batches = (S + 63) / 64;
    const NearBatch* batches = a.batches + a.batch_ptr[leaf];
    double* st = lds + w * F::kStage;
    const int need = (tc + R - 1) / R;
    int L = 1;
    while (L < need) L <<= 1;
    const int G = 64 / L, li = lane & (L - 1), g = lane / L;
    typename F::Pos t[R];
    double sum[R][NS];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int it = item.target + min(li + r * L, tc - 1);
        t[r] = f.pos(a.X[it] - cx, a.Y[it] - cy, a.Z[it] - cz);
#pragma unroll
        for (int c = 0; c < NS; ++c) sum[r][c] = 0.0;
    }
    // of batch b (clamped to the last): the record, the lane's shift from source to point, the point
    auto record = [&](int b) { return batches[min(b, n_batches - 1)]; };
    auto source = [&](int b) { return min(64 * min(b, n_batches - 1) + lane, S - 1); };
    auto shift = [&](int b, const NearBatch& rec) {
        const int i = source(b) & 63;
        return a.rng_delta[rec.first + __popcll(rec.mask & (~0ull >> (63 - i)))];
    };
    const int b0 = w;
    NearBatch rec = record(b0);
    int sh = shift(b0, rec);
    rec = record(b0 + kNearWaves);
    int idx = source(b0) + sh;
    double x = a.X[idx], y = a.Y[idx], z = a.Z[idx];
    double2 q = a.q[idx];
    sh = shift(b0 + kNearWaves, rec);
    rec = record(b0 + 2 * kNearWaves);
    for (int b = b0; b < n_batches; b += kNearWaves) {
        const bool odd = F::kSkips && __ballot(!nearfield::finite_charge(q.x, q.y)) != 0;
        f.stage(st, lane, x - cx, y - cy, z - cz, q);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        idx = source(b + kNearWaves) + sh;
        x = a.X[idx];
        y = a.Y[idx];
        z = a.Z[idx];
        q = a.q[idx];
        sh = shift(b + 2 * kNearWaves, rec);
        rec = record(b + 3 * kNearWaves);
        typename F::Acc acc[R][NS];
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < NS; ++c) acc[r][c] = 0;
        const int n = min(64, S - 64 * b);
        if (odd) {
            if constexpr (F::kSkips)
                for (int j = g; j < n; j += G) {
                    const typename F::Src s = f.load(st, j);
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (f.apart(t[r], s)) f.pair(t[r], s, acc[r]);
                }
        } else {
            for (int j = g; j < n; j += G) {
                const typename F::Src s = f.load(st, j);
#pragma unroll
                for (int r = 0; r < R; ++r) f.pair(t[r], s, acc[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < NS; ++c) sum[r][c] += (double)acc[r][c];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
    for (int off = L; off < 64; off <<= 1)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < NS; ++c) sum[r][c] += __shfl_xor(sum[r][c], off);
    // the waves' sums, per wave [sum c][target]
    __syncthreads();
    if (g == 0)
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int c = 0; c < NS; ++c) lds[(w * NS + c) * (64 * R) + li + r * L] = sum[r][c];
    __syncthreads();
    for (int i = threadIdx.x; i < tc * (NS / 2); i += kNearThreads) {
        const int ti = i % tc, c = i / tc, it = item.target + ti;
        double2 v = make_double2(0.0, 0.0);
#pragma unroll
        for (int u = 0; u < kNearWaves; ++u) {
            v.x += lds[(u * NS + 2 * c) * (64 * R) + ti];
            v.y += lds[(u * NS + 2 * c + 1) * (64 * R) + ti];
        }
        const int o = a.perm[it];
        const double2 far = c ? a.far_e[3 * (int64_t)it + c - 1] : a.far[it];
        v.x = fma(v.x, a.wscale, far.x);
        v.y = fma(v.y, a.wscale, far.y);
        v = out_value(v, a.out_mode);
        if (c)
            a.field[3 * (int64_t)o + c - 1] = v;
        else
            a.out[o] = v;
    }
}

// The FP32-phase leaves take the FP32 coordinates where the leaf is flagged
template <class F, int R>
__device__ __forceinline__ void near_item(const P2PArgs& a, const NearItem item, double* lds) {
    if (item.n_targets == 0) return;   // padding
    if constexpr (std::is_same<F, FormMixed<false, false>>::value) {
        if (a.coord32 && a.coord32[item.leaf]) {   // uniform
            near_body<FormMixed32, R>(a, item, lds);
            return;
        }
    }
    near_body<F, R>(a, item, lds);
}

// workgroup i runs on XCD i % 8, whose items are every 8th of the list
template <class F, int R>
__global__ __launch_bounds__(kNearThreads) void near_kernel(P2PArgs a, const NearItem* __restrict__ items) {
    __shared__ __attribute__((aligned(16))) double lds[near_lds_doubles<F, R>()];
    near_item<F, R>(a, items[blockIdx.x], lds);
}

// items of many problems in one launch: args[prob[i]] describes the problem of item i
template <class F, int R>
__global__ __launch_bounds__(kNearThreads) void near_batch_kernel(const P2PArgs* __restrict__ args,
                                                                  const NearItem* __restrict__ items,
                                                                  const int* __restrict__ prob) {
    __shared__ __attribute__((aligned(16))) double lds[near_lds_doubles<F, R>()];
    const P2PArgs a = args[prob[blockIdx.x]];
    near_item<F, R>(a, items[blockIdx.x], lds);
}

// Setup: the estimate of a leaf's error from FP32 coordinates (launch_p2p_coord_check).  One wave per leaf
// of the FP32 phase: lane t holds target t of a 64-target chunk and scans every source of the leaf
// (uniform loads), FP64 throughout.
__global__ __launch_bounds__(64) void p2p_coord_check_kernel(P2PArgs a, double tol, unsigned char* flag) {
    const int leaf = blockIdx.x;
    const int b = a.leaf_box[leaf];
    const int tstart = a.bx.pstart[b], tcnt = a.bx.count[b];
    const double cx = a.bx.centre[3 * b], cy = a.bx.centre[3 * b + 1], cz = a.bx.centre[3 * b + 2];
    const int S = a.leaf_src_total[leaf];
    const NearBatch* batches = a.batches + a.batch_ptr[leaf];
    const double fl2 = a.floor2[leaf];
    const int lane = threadIdx.x;
    double cmax = 0.0, ratio = 0.0;
    for (int t0 = 0; t0 < tcnt; t0 += 64) {
        const bool has = t0 + lane < tcnt;
        const int it = tstart + t0 + (has ? lane : 0);
        const double xt = a.X[it] - cx, yt = a.Y[it] - cy, zt = a.Z[it] - cz;
        if (has) cmax = fmax(cmax, fmax(fabs(xt), fmax(fabs(yt), fabs(zt))));
        double s2 = 0.0, s4 = 0.0;
        for (int v = 0; v < S; ++v) {
            const NearBatch rec = batches[v / 64];
            const int idx = v + a.rng_delta[rec.first + __popcll(rec.mask & (~0ull >> (63 - v % 64)))];
            const double xs = a.X[idx] - cx, ys = a.Y[idx] - cy, zs = a.Z[idx] - cz;
            if (t0 == 0) cmax = fmax(cmax, fmax(fabs(xs), fmax(fabs(ys), fabs(zs))));
            const double dx = xt - xs, dy = yt - ys, dz = zt - zs;
            const double r2 = dx * dx + dy * dy + dz * dz;
            if (r2 > fl2) {
                const double w = 1.0 / r2;
                s2 += w;
                s4 += w * w;
            }
        }
        if (has && s2 > 0.0) ratio = fmax(ratio, sqrt(s4 / s2));
    }
    for (int off = 1; off < 64; off <<= 1) {
        cmax = fmax(cmax, __shfl_xor(cmax, off));
        ratio = fmax(ratio, __shfl_xor(ratio, off));
    }
    if (lane == 0) flag[leaf] = 0x1p-21 * cmax * ratio <= tol ? 1 : 0;
}

template <class F, int R>
void launch_form(const P2PArgs& a, const NearItems& it, hipStream_t s) {
    if (it.n > 0) hipLaunchKernelGGL((near_kernel<F, R>), dim3(it.n), dim3(kNearThreads), 0, s, a, it.items);
}

template <int R>
void launch_mixed(const P2PArgs& a, const NearItems* items, bool lowk, hipStream_t s) {
    if (lowk) {
        launch_form<FormMixed<false, true>, R>(a, items[0], s);
        return;
    }
    launch_form<FormMixed<false, false>, R>(a, items[0], s);
    launch_form<FormMixed<true, false>, R>(a, items[1], s);
}

void check_launch(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) fail(-3, std::string("kernel launch failed (") + what + "): " + hipGetErrorString(e));
}

}  // namespace

P2PArgs p2p_scaled(P2PArgs a, int precision, bool lowk) {
    // coordinates in units of pi / k: the weights are e^{i pi u}/u with u = k r / pi
    a.scale = a.wscale = precision == 0 || lowk ? 1.0 : a.k / M_PI;
    return a;
}

void launch_p2p(const P2PArgs& a0, const NearItems* items, int precision, bool lowk, int tile, hipStream_t s) {
    const P2PArgs a = p2p_scaled(a0, precision, lowk);
    if (precision == 0)
        launch_form<FormFp64, kP2PFp64TargetsPerLane>(a, items[0], s);
    else if (tile == 1)
        launch_mixed<1>(a, items, lowk, s);
    else if (tile == 4)
        launch_mixed<4>(a, items, lowk, s);
    else
        launch_mixed<2>(a, items, lowk, s);
    check_launch("p2p");
}

void launch_p2p_field(const P2PArgs& a0, const NearItems* items, int precision, hipStream_t s) {
    P2PArgs a = a0;
    a.wscale = 1.0;
    if (precision == 0) {
        launch_form<FormField<double, false>, 1>(a, items[0], s);
    } else {
        launch_form<FormField<float, false>, 1>(a, items[0], s);
        launch_form<FormField<float, true>, 1>(a, items[1], s);
    }
    check_launch("p2p_field");
}

void launch_p2p_batch(int cls, const P2PArgs* d_args, const NearItem* items, const int* prob, int n, hipStream_t s) {
    if (n <= 0) return;
    auto go = [&](auto k) { hipLaunchKernelGGL(k, dim3(n), dim3(kNearThreads), 0, s, d_args, items, prob); };
    constexpr int R = kP2PBatchTargetsPerLane;
    if (cls == kP2PClassFp64)
        go(near_batch_kernel<FormFp64, kP2PFp64TargetsPerLane>);
    else if (cls == kP2PClassLowK)
        go(near_batch_kernel<FormMixed<false, true>, R>);
    else if (cls == kP2PClassPhase32)
        go(near_batch_kernel<FormMixed<false, false>, R>);
    else
        go(near_batch_kernel<FormMixed<true, false>, R>);
    check_launch("p2p batch");
}

void launch_p2p_coord_check(const P2PArgs& a, int n, double tol, unsigned char* flag, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(p2p_coord_check_kernel, dim3(n), dim3(64), 0, s, a, tol, flag);
    check_launch("p2p coordinate check");
}
}  // namespace hfmm
