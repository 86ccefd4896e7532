// M2L in FP32 on matrix cores, one wave per work item and one matrix column per lane.
//
// Basis, groups and work items are those of the FP64 kernel (m2l_wave64.hip): S and D halves, pairs (target
// box, source box) of equal polar angle and length, partial sums for split blocks.  Here a group is 32 pairs,
// and lane 2 c + j holds the real (j = 0) or imaginary (j = 1) part of every S or u entry of pair c, and the
// other part of every D or v entry: u = c S + i s D and v = c D + i s S then need no exchange between lanes.
// Every product is a chain of 4 x 4 x 1 MFMAs of 16 blocks: their 64 columns are the lanes, a B operand is one
// entry of the lane's column in one register, and the A operand, a column of four operator entries, is the
// same for all blocks (cbsz = 4 broadcasts the block `abid` of a register, so that one register holds 16 such
// columns and a 16-byte load 64 of them). Compared with 16 x 16 x 4 tiles the inner dimension needs no padding
// and the rows are padded to four, and no data moves between lanes but the exchange of real and imaginary
// parts for the complex coaxial products (DPP).  Per group and half, u, then v:
//   1. per degree n: the source's S and D entries (loaded straight into registers) times e^{i m phi}
//      are the inputs of the forward rotation; its results go to LDS, which serves as a register
//      extension: a lane reads its own column only;
//   2. per order m: coaxial operator, in place;
//   3. per degree n: back rotation, times e^{-i m phi}, added to the U and V accumulators.
// Operator columns, sources and phases are fetched ahead, those of the next group during this one.
// Up to degree 11 the two halves go one after the other (wave32_split_body), which lets two waves fit a
// SIMD; above, one wave per SIMD takes both at once (wave32_joint_body), each with its layout of the
// operators (p = 11: split 1.81 ms, joint 1.97 on 5.4M pairs; p = 12: split 0.366, joint 0.329 on 584136).
// Bound by the issue of MFMA and VALU instructions, which do not overlap on this chip (1358 MFMAs of 8 cycles
// and 744 VALU instructions per group at p = 11: 50% and 14% of the time on 5.4M pairs, 43% and 13% at p = 12,
// one wave per SIMD), and by what the latencies leave exposed.  Against the block kernel (16 x 16 x 4 tiles,
// 16 targets x 2 directions per workgroup): 5.4M pairs at p = 11 3.96 -> 1.65 ms with the sums, 584136 at p =
// 12 0.84 -> 0.325, 53352 at p = 14 0.19 -> 0.077; the five levels of 100k points (p = 11) 1.39 -> 0.33 ms, of
// 300k on surfaces (p = 10) 2.3 -> 0.52, of 150k at k = 0 (p = 7) 0.52 -> 0.136.  Errors against FP64 are
// those of the block kernel (1.1e-7 to 1.6e-7 of the potential).
#include <hip/hip_runtime.h>

#include <string>
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace hfmm {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) int* ScalarInts;   // uniform loads: scalar cache

__host__ __device__ constexpr int tri(int n) { return n * (n + 1) / 2; }
constexpr int quads(int n) { return (n + 3) / 4; }

// c + A B: A the four operator entries of block ABID of register a, B the lanes' entries b
template <int ABID>
__device__ __forceinline__ f4 mma(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 4, ABID, 0);
}

// the value of the lane that holds the other part of the pair
__device__ __forceinline__ float other(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xF, 0xF, true));
}

template <int A, int B, typename F>
__device__ __forceinline__ void unrolled(F&& f) {
    if constexpr (A < B) {
        f(std::integral_constant<int, A>{});
        unrolled<A + 1, B>(f);
    }
}
#define IDX(x) decltype(x)::value

// row of (degree n, order m) of half h in the lane's column: u_0..u_n or v_1..v_n, degrees in order
constexpr int row(int h, int n, int m) { return h ? tri(n - 1) + m - 1 : tri(n) + m; }
// U and V parts (real for even lanes) of degree n and order m stored in the x basis: x_0 = U_0,
// x_m = (U + V) / 2, x_{-m} = (-1)^m (U - V) / 2
__device__ __forceinline__ void store_expansion(double* dst, int n, int m, double u, double v) {
    const double sg = (m & 1) ? -0.5 : 0.5;
    dst[2 * (n * n + n + m)] = m == 0 ? u : 0.5 * (u + v);
    if (m > 0) dst[2 * (n * n + n - m)] = sg * (u - v);
}

// row of (degree n, half h, order m) in the lane's column, degrees in order: u_0..u_n, v_1..v_n
constexpr int joint_row(int n, int h, int m) { return n * n + (h ? n + m : m); }
// rows of a column in LDS, so that four waves fit a compute unit's 160 KiB; the rest, the lowest
// degrees, stay in registers
constexpr int kLdsRows = 160;
constexpr int reg_rows(int P) { return (P + 1) * (P + 1) > kLdsRows ? (P + 1) * (P + 1) - kLdsRows : 0; }
__host__ __device__ constexpr int joint_lds_bytes(int P) { return 256 * ((P + 1) * (P + 1) < kLdsRows ? (P + 1) * (P + 1) : kLdsRows); }

// The columns of a target (pairs c = target mod tb) added, then stored
template <int P>
__device__ __forceinline__ void store_item(const M2LWaveArgs& a, const int4 item, float* U, float* V) {
    constexpr int NU = tri(P + 1), NV = tri(P);
    const int lane = threadIdx.x, c = lane >> 1;
    const int tb = a.tb;
    unrolled<0, NV>([&](auto ic) { V[IDX(ic)] = other(V[IDX(ic)]); });
    for (int off = 2 * tb; off < 64; off <<= 1) {
        const int from = (lane ^ off) << 2;
        auto fold = [&](float& v) { v += __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(v))); };
        unrolled<0, NU>([&](auto ic) { fold(U[IDX(ic)]); });
        unrolled<0, NV>([&](auto ic) { fold(V[IDX(ic)]); });
    }
    if (lane >= 2 * tb) return;
    if (item.w > 0) {   // one of several parts of the block: summed by wave32_sum_kernel
        float* part = (float*)a.part + (size_t)(item.w - 1) * (NU + NV) * (2 * tb) + lane;
        unrolled<0, NU>([&](auto ic) { part[IDX(ic) * 2 * tb] = U[IDX(ic)]; });
        unrolled<0, NV>([&](auto ic) { part[(NU + IDX(ic)) * 2 * tb] = V[IDX(ic)]; });
        return;
    }
    const int tbox = a.blk_targets[(size_t)item.x * tb + c];
    if (tbox < 0) return;
    double* dst = (double*)(a.L + a.exp_off[tbox]) + (lane & 1);
    unrolled<0, P + 1>([&](auto nc) {
        unrolled<0, IDX(nc) + 1>([&](auto mc) {
            constexpr int n = IDX(nc), m = IDX(mc), iv = m ? tri(n - 1) + m - 1 : 0;
            store_expansion(dst, n, m, U[tri(n) + m], m ? V[iv] : 0.0f);
        });
    });
}

// One work item (block, first group, end group, part) at degree P, u and v together
template <int P, int kFragAhead, int kGatherAhead>
__device__ __forceinline__ void wave32_joint_body(const M2LWaveArgs& a, const int4 item) {
    extern __shared__ float lds32[];
    constexpr int NU = tri(P + 1), NV = tri(P), NP = (NU + 1) / 2;
    constexpr int RK = reg_rows(P);
    constexpr int BR = (wave32_joint_vecs(P + 1) + 63) / 64, BC = (wave32_coax_vecs(P, P + 1) + 63) / 64;
    constexpr int NB = 2 * BR + BC, RING = kFragAhead + 1, GA = kGatherAhead < NP ? kGatherAhead : NP;
    if (item.y >= item.z) return;   // padding item
    const int lane = threadIdx.x, c = lane >> 1;
    const float sgn = (lane & 1) ? 1.0f : -1.0f;
    float* const X = lds32 + lane;
    float xr[RK > 0 ? RK : 1];
    auto put = [&](auto rc, float v) {
        constexpr int r = IDX(rc);
        if constexpr (r < RK)
            xr[r] = v;
        else
            X[64 * (r - RK)] = v;
    };
    auto get = [&](auto rc) -> float {
        constexpr int r = IDX(rc);
        if constexpr (r < RK)
            return xr[r];
        else
            return X[64 * (r - RK)];
    };
    float U[NU], V[NV];   // [tri(n) + m], [tri(n - 1) + m - 1]
    unrolled<0, NU>([&](auto ic) { U[IDX(ic)] = 0.0f; });
    unrolled<0, NV>([&](auto ic) { V[IDX(ic)] = 0.0f; });

    const uint32_t lane16 = 16 * (uint32_t)lane;
    const float *R1, *R3, *T;
    auto operators = [&](int cls) {   // theta | dist << 16
        R1 = (const float*)a.rot1 + (size_t)(cls & 0xFFFF) * a.rot_stride;
        R3 = (const float*)a.rot3 + (size_t)(cls & 0xFFFF) * a.rot_stride;
        T = (const float*)a.coax + (size_t)(cls >> 16) * a.coax_stride;
    };
    // block b of 64 operator columns: forward rotations, coaxial operators, back rotations
    f4 fr[RING];
    auto frag_load = [&](auto bc) {
        constexpr int b = IDX(bc), st = b < BR ? 0 : b < BR + BC ? 1 : 2, o = st == 0 ? b : st == 1 ? b - BR : b - BR - BC;
        fr[b % RING] = *(const f4*)((const char*)((st == 0 ? R1 : st == 1 ? T : R3) + 256 * o) + lane16);
    };
    // Y += column v of stage st times b
    auto madd = [&](auto sc, auto vc, float b, f4& y) {
        constexpr int st = IDX(sc), v = IDX(vc), blk = (st == 0 ? 0 : st == 1 ? BR : BR + BC) + v / 64;
        y = mma<v % 16>(fr[blk % RING][(v % 64) / 16], b, y);
    };
    // the first column of a block frees the block before the last but kFragAhead
    auto advance = [&](auto sc, auto vc) {
        constexpr int st = IDX(sc), v = IDX(vc), blk = (st == 0 ? 0 : st == 1 ? BR : BR + BC) + v / 64;
        if constexpr (v % 64 == 0 && blk + kFragAhead < NB) frag_load(std::integral_constant<int, blk + kFragAhead>{});
    };
    // pair i of the source's entries: S, D, S, D (D the other part of the pair's than S)
    f4 g[GA];
    uint32_t so;
    const uint32_t ri = 16 * (uint32_t)(lane & 1);   // the lane's parts of a pair
    auto gather_load = [&](auto ic) {
        constexpr int i = IDX(ic);
        g[i % GA] = *(const f4*)((const char*)a.M + 32 * i + so);
    };
    float cp[P + 1], tp[P + 1];   // cos m phi; -sin m phi (even lanes), sin m phi (odd)
    float2 phn[P + 1];
    auto phase_load = [&](int dir) {
        unrolled<1, P + 1>([&](auto mc) {
            constexpr int m = IDX(mc);
            phn[m] = ((const float2*)a.phase)[(size_t)dir * a.phase_stride + min(m, a.phase_stride - 1)];
        });
    };
    int src = a.grp_src[(size_t)item.y * 32 + c], dir = a.grp_dir[(size_t)item.y * 32 + c];
    operators(((ScalarInts)a.grp_class)[item.y]);
    so = 32 * (uint32_t)src + ri;
    unrolled<0, GA>(gather_load);
    phase_load(dir);
    unrolled<0, kFragAhead>([&](auto bc) {
        if constexpr (IDX(bc) < NB) frag_load(bc);
    });
#pragma unroll 1
    for (int e = item.y; e < item.z; ++e) {
        unrolled<1, P + 1>([&](auto mc) {
            constexpr int m = IDX(mc);
            cp[m] = phn[m].x;
            tp[m] = sgn * phn[m].y;
        });
        const int en = e + 1 < item.z ? e + 1 : e;
        src = a.grp_src[(size_t)en * 32 + c];
        dir = a.grp_dir[(size_t)en * 32 + c];
        const int cls = ((ScalarInts)a.grp_class)[en];
        f4 yu[2][4], yv[2][4];
        auto clear = [&](auto qc, auto nq) {
            unrolled<0, IDX(nq)>([&](auto rc) {
                yu[IDX(qc)][IDX(rc)] = f4{0, 0, 0, 0};
                yv[IDX(qc)][IDX(rc)] = f4{0, 0, 0, 0};
            });
        };
        // rotation of degree n (stage st): inputs u[0..n], v[1..n]
        auto rotate = [&](auto sc, auto nc, const float* u, const float* v) {
            constexpr int n = IDX(nc), qu = quads(n + 1), qv = quads(n), base = wave32_joint_vecs(n);
            clear(std::integral_constant<int, (n & 1)>{}, std::integral_constant<int, qu>{});
            unrolled<0, n + 1>([&](auto kc) {
                constexpr int k = IDX(kc), o = base + k * qu + (k ? (k - 1) * qv : 0);
                unrolled<0, qu>([&](auto rc) {
                    constexpr std::integral_constant<int, o + IDX(rc)> vc;
                    advance(sc, vc);
                    madd(sc, vc, u[k], yu[n & 1][IDX(rc)]);
                });
                if constexpr (k > 0)
                    unrolled<0, qv>([&](auto rc) {
                        constexpr std::integral_constant<int, o + qu + IDX(rc)> vc;
                        advance(sc, vc);
                        madd(sc, vc, v[k], yv[n & 1][IDX(rc)]);
                    });
            });
        };

        // 1. phases and forward rotations
        auto finish1 = [&](auto nc) {
            constexpr int n = IDX(nc);
            unrolled<0, n + 1>([&](auto mc) {
                constexpr int m = IDX(mc);
                put(std::integral_constant<int, joint_row(n, 0, m)>{}, yu[n & 1][m / 4][m % 4]);
                if constexpr (m > 0) put(std::integral_constant<int, joint_row(n, 1, m)>{}, yv[n & 1][(m - 1) / 4][(m - 1) % 4]);
            });
        };
        unrolled<0, P + 1>([&](auto nc) {
            constexpr int n = IDX(nc);
            float u[n + 1], v[n + 1];
            unrolled<0, n + 1>([&](auto mc) {
                constexpr int m = IDX(mc), i = tri(n) + m;
                const f4 w = g[(i / 2) % GA];
                const float S = (i & 1) ? w.z : w.x, D = (i & 1) ? w.w : w.y;
                if constexpr (m == 0) {
                    u[0] = S;
                } else {
                    u[m] = fmaf(tp[m], D, cp[m] * S);
                    v[m] = fmaf(-tp[m], S, cp[m] * D);
                }
                if constexpr (((i & 1) || i == NU - 1) && i / 2 + GA < NP) gather_load(std::integral_constant<int, i / 2 + GA>{});
            });
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (n == 0) {
                put(std::integral_constant<int, 0>{}, u[0]);
            } else {
                if constexpr (n > 1) finish1(std::integral_constant<int, n - 1>{});
                rotate(std::integral_constant<int, 0>{}, nc, u, v);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        finish1(std::integral_constant<int, P>{});

        // 2. coaxial operators; the rows of the next order are read before this one's products
        so = 32 * (uint32_t)src + ri;
        float xu[2][P + 1], xv[2][P + 1];
        auto rows2 = [&](auto mc) {
            constexpr int m = IDX(mc);
            unrolled<m, P + 1>([&](auto nc) {
                constexpr int n = IDX(nc);
                xu[m & 1][n - m] = get(std::integral_constant<int, joint_row(n, 0, m)>{});
                if constexpr (m > 0) xv[m & 1][n - m] = get(std::integral_constant<int, joint_row(n, 1, m)>{});
            });
        };
        auto finish2 = [&](auto mc) {
            constexpr int m = IDX(mc);
            unrolled<m, P + 1>([&](auto nc) {
                constexpr int n = IDX(nc);
                put(std::integral_constant<int, joint_row(n, 0, m)>{}, yu[m & 1][(n - m) / 4][(n - m) % 4]);
                if constexpr (m > 0) put(std::integral_constant<int, joint_row(n, 1, m)>{}, yv[m & 1][(n - m) / 4][(n - m) % 4]);
            });
        };
        rows2(std::integral_constant<int, 0>{});
        unrolled<0, P + 1>([&](auto mc) {
            constexpr int m = IDX(mc), L = P + 1 - m, q = quads(L), base = wave32_coax_vecs(P, m);
            constexpr std::integral_constant<int, 1> sc;
            if constexpr (m < P) rows2(std::integral_constant<int, m + 1>{});
            float zu[L], zv[L];   // i x (v's parts are exchanged)
            unrolled<0, L>([&](auto kc) {
                constexpr int k = IDX(kc);
                zu[k] = sgn * other(xu[m & 1][k]);
                if constexpr (m > 0) zv[k] = -sgn * other(xv[m & 1][k]);
            });
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (m > 0) finish2(std::integral_constant<int, m - 1>{});
            clear(std::integral_constant<int, (m & 1)>{}, std::integral_constant<int, q>{});
            unrolled<0, L>([&](auto kc) {
                constexpr int k = IDX(kc);
                unrolled<0, 2 * q>([&](auto rc) {
                    constexpr int r = IDX(rc) % q, im = IDX(rc) / q;
                    constexpr std::integral_constant<int, base + 2 * q * k + IDX(rc)> vc;
                    advance(sc, vc);
                    madd(sc, vc, im ? zu[k] : xu[m & 1][k], yu[m & 1][r]);
                    if constexpr (m > 0) madd(sc, vc, im ? zv[k] : xv[m & 1][k], yv[m & 1][r]);
                });
            });
            __builtin_amdgcn_sched_barrier(0);
        });
        finish2(std::integral_constant<int, P>{});

        // 3. back rotations and phases; the next group's first entries and phases are on their way
        auto rows3 = [&](auto nc) {
            constexpr int n = IDX(nc);
            unrolled<0, n + 1>([&](auto mc) {
                constexpr int m = IDX(mc);
                xu[n & 1][m] = get(std::integral_constant<int, joint_row(n, 0, m)>{});
                if constexpr (m > 0) xv[n & 1][m] = get(std::integral_constant<int, joint_row(n, 1, m)>{});
            });
        };
        auto finish3 = [&](auto nc) {
            constexpr int n = IDX(nc);
            unrolled<0, n + 1>([&](auto mc) {
                constexpr int m = IDX(mc);
                const float yum = yu[n & 1][m / 4][m % 4];
                float& A = U[tri(n) + m];
                if constexpr (m == 0) {
                    A += yum;
                    asm volatile("" : "+v"(A));
                } else {
                    const float yvm = yv[n & 1][(m - 1) / 4][(m - 1) % 4];
                    float& B = V[tri(n - 1) + m - 1];
                    A = fmaf(-tp[m], yvm, fmaf(cp[m], yum, A));
                    B = fmaf(tp[m], yum, fmaf(cp[m], yvm, B));
                    // computed here: sunk to the end of the group, the products would stay live
                    asm volatile("" : "+v"(A), "+v"(B));
                }
            });
        };
        U[0] += get(std::integral_constant<int, 0>{});
        rows3(std::integral_constant<int, 1>{});
        unrolled<0, GA>(gather_load);
        phase_load(dir);
        __builtin_amdgcn_sched_barrier(0);
        unrolled<1, P + 1>([&](auto nc) {
            constexpr int n = IDX(nc);
            if constexpr (n < P) rows3(std::integral_constant<int, n + 1>{});
            rotate(std::integral_constant<int, 2>{}, nc, xu[n & 1], xv[n & 1]);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (n > 1) finish3(std::integral_constant<int, n - 1>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        operators(cls);
        unrolled<0, kFragAhead>([&](auto bc) {
            if constexpr (IDX(bc) < NB) frag_load(bc);
        });
        finish3(std::integral_constant<int, P>{});
    }

    store_item<P>(a, item, U, V);
}

// The same, u, then v: half the rows in LDS and half the registers in flight, for the degrees at
// which two waves then fit a SIMD; the sources' entries and the coaxial operators are read twice
template <int P, int kFragAhead, int kGatherAhead>
__device__ __forceinline__ void wave32_split_body(const M2LWaveArgs& a, const int4 item) {
    extern __shared__ float lds32[];
    constexpr int NU = tri(P + 1), NV = tri(P), NP = (NU + 1) / 2;
    constexpr int RING = kFragAhead + 1, GA = kGatherAhead < NP ? kGatherAhead : NP;
    if (item.y >= item.z) return;   // padding item
    const int lane = threadIdx.x, c = lane >> 1;
    const float sgn = (lane & 1) ? 1.0f : -1.0f;
    float* const X = lds32 + lane;
    float U[NU], V[NV];   // [tri(n) + m], [tri(n - 1) + m - 1]
    unrolled<0, NU>([&](auto ic) { U[IDX(ic)] = 0.0f; });
    unrolled<0, NV>([&](auto ic) { V[IDX(ic)] = 0.0f; });

    const uint32_t lane16 = 16 * (uint32_t)lane;
    const float *R1, *R3, *T;
    auto operators = [&](int cls) {   // theta | dist << 16
        R1 = (const float*)a.rot1 + (size_t)(cls & 0xFFFF) * a.rot_stride;
        R3 = (const float*)a.rot3 + (size_t)(cls & 0xFFFF) * a.rot_stride;
        T = (const float*)a.coax + (size_t)(cls >> 16) * a.coax_stride;
    };
    f4 fr[RING], g[GA];
    // pair i of the source's entries: S, D, S, D (D the other part of the pair's than S)
    uint32_t so;
    const uint32_t ri = 16 * (uint32_t)(lane & 1);   // the lane's parts of a pair
    auto gather_load = [&](auto ic) {
        constexpr int i = IDX(ic);
        g[i % GA] = *(const f4*)((const char*)a.M + 32 * i + so);
    };
    // block b of 64 operator columns of half h: forward rotations, coaxial operators, back rotations
    auto frag_load = [&](auto hc, auto bc) {
        constexpr int h = IDX(hc), b = IDX(bc), BR = wave32_blocks(wave32_rot_vecs(h, P + 1));
        constexpr int B0 = wave32_coax_vecs(P, h) / 64, BC = wave32_blocks(wave32_coax_vecs(P, P + 1)) - B0;
        constexpr int st = b < BR ? 0 : b < BR + BC ? 1 : 2;
        constexpr int o = st == 1 ? b - BR + B0 : (h ? kWave32VBlock : 0) + (st == 0 ? b : b - BR - BC);
        fr[b % RING] = *(const f4*)((const char*)((st == 0 ? R1 : st == 1 ? T : R3) + 256 * o) + lane16);
    };
    float cp[P + 1], tp[P + 1];   // cos m phi; -sin m phi (even lanes), sin m phi (odd)
    float2 phn[P + 1];
    auto phase_load = [&](int dir) {
        unrolled<1, P + 1>([&](auto mc) {
            constexpr int m = IDX(mc);
            phn[m] = ((const float2*)a.phase)[(size_t)dir * a.phase_stride + min(m, a.phase_stride - 1)];
        });
    };
    int src = a.grp_src[(size_t)item.y * 32 + c], dir = a.grp_dir[(size_t)item.y * 32 + c];
    operators(((ScalarInts)a.grp_class)[item.y]);
    so = 32 * (uint32_t)src + ri;
    unrolled<0, GA>(gather_load);
    unrolled<0, kFragAhead>([&](auto bc) { frag_load(std::integral_constant<int, 0>{}, bc); });
#pragma unroll 1
    for (int e = item.y; e < item.z; ++e) {
        phase_load(dir);
        unrolled<1, P + 1>([&](auto mc) {
            constexpr int m = IDX(mc);
            cp[m] = phn[m].x;
            tp[m] = sgn * phn[m].y;
        });
        const int en = e + 1 < item.z ? e + 1 : e;
        src = a.grp_src[(size_t)en * 32 + c];
        dir = a.grp_dir[(size_t)en * 32 + c];
        const int cls = ((ScalarInts)a.grp_class)[en];
        unrolled<0, 2>([&](auto hc) {
            // blocks of a rotation; first block of the coaxial operators from order h, and their blocks
            constexpr int h = IDX(hc), BR = wave32_blocks(wave32_rot_vecs(h, P + 1));
            constexpr int V0 = wave32_coax_vecs(P, h), B0 = V0 / 64, BC = wave32_blocks(wave32_coax_vecs(P, P + 1)) - B0;
            constexpr int NB = 2 * BR + BC;
            f4 y[2][4];
            float x[2][P + 1];
            auto clear = [&](auto ic, auto qc) {
                unrolled<0, IDX(qc)>([&](auto rc) { y[IDX(ic) & 1][IDX(rc)] = f4{0, 0, 0, 0}; });
            };
            // Y += column v of stage st times b; the first column of a block frees the one before
            auto madd = [&](auto sc, auto vc, float b, f4& Y) {
                constexpr int st = IDX(sc), v = IDX(vc), blk = (st == 0 ? 0 : st == 1 ? BR - B0 : BR + BC) + v / 64;
                if constexpr ((v % 64 == 0 || (st == 1 && v == V0)) && blk + kFragAhead < NB) frag_load(hc, std::integral_constant<int, blk + kFragAhead>{});
                Y = mma<v % 16>(fr[blk % RING][(v % 64) / 16], b, Y);
            };
            // rotation of degree n (stage st): inputs in[m - h], m = h..n
            auto rotate = [&](auto sc, auto nc, const float* in) {
                constexpr int n = IDX(nc), L = n + 1 - h, q = quads(L);
                clear(nc, std::integral_constant<int, q>{});
                unrolled<0, L * q>([&](auto ic) {
                    constexpr int i = IDX(ic);
                    madd(sc, std::integral_constant<int, wave32_rot_vecs(h, n) + i>{}, in[i / q], y[n & 1][i % q]);
                });
            };
            auto put_rows = [&](auto nc) {   // results of the forward rotation of degree n
                constexpr int n = IDX(nc);
                unrolled<h, n + 1>([&](auto mc) {
                    constexpr int m = IDX(mc);
                    X[64 * row(h, n, m)] = y[n & 1][(m - h) / 4][(m - h) % 4];
                });
            };
            auto get_rows = [&](auto nc) {   // inputs of the back rotation of degree n
                constexpr int n = IDX(nc);
                unrolled<h, n + 1>([&](auto mc) { x[n & 1][IDX(mc) - h] = X[64 * row(h, n, IDX(mc))]; });
            };
            auto put_order = [&](auto mc) {
                constexpr int m = IDX(mc);
                unrolled<m, P + 1>([&](auto nc) { X[64 * row(h, IDX(nc), m)] = y[m & 1][(IDX(nc) - m) / 4][(IDX(nc) - m) % 4]; });
            };
            auto get_order = [&](auto mc) {
                constexpr int m = IDX(mc);
                unrolled<m, P + 1>([&](auto nc) { x[m & 1][IDX(nc) - m] = X[64 * row(h, IDX(nc), m)]; });
            };

            // 1. phases and forward rotations
            unrolled<0, P + 1>([&](auto nc) {
                constexpr int n = IDX(nc);
                float in[n + 1];
                unrolled<0, n + 1>([&](auto mc) {
                    constexpr int m = IDX(mc), i = tri(n) + m;
                    const f4 w = g[(i / 2) % GA];
                    const float S = (i & 1) ? w.z : w.x;
                    const float D = (i & 1) ? w.w : w.y;
                    if constexpr (m > 0) {
                        in[m - h] = h ? fmaf(-tp[m], S, cp[m] * D) : fmaf(tp[m], D, cp[m] * S);
                    } else if constexpr (h == 0) {
                        in[0] = S;
                    }
                    if constexpr (((i & 1) || i == NU - 1) && i / 2 + GA < NP) gather_load(std::integral_constant<int, i / 2 + GA>{});
                });
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (n == 0) {
                    if constexpr (h == 0) X[0] = in[0];
                } else {
                    if constexpr (n > 1) put_rows(std::integral_constant<int, n - 1>{});
                    rotate(std::integral_constant<int, 0>{}, nc, in);
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            put_rows(std::integral_constant<int, P>{});

            // 2. coaxial operators; the rows of the next order are read before this one's products
            get_order(hc);
            unrolled<h, P + 1>([&](auto mc) {
                constexpr int m = IDX(mc), L = P + 1 - m, q = quads(L), base = wave32_coax_vecs(P, m);
                if constexpr (m < P) get_order(std::integral_constant<int, m + 1>{});
                float z[L];   // i x (v's parts are exchanged)
                unrolled<0, L>([&](auto kc) { z[IDX(kc)] = (h ? -sgn : sgn) * other(x[m & 1][IDX(kc)]); });
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (m > h) put_order(std::integral_constant<int, m - 1>{});
                clear(mc, std::integral_constant<int, q>{});
                unrolled<0, 2 * L * q>([&](auto ic) {
                    constexpr int i = IDX(ic), k = i / (2 * q), im = i / q % 2;
                    madd(std::integral_constant<int, 1>{}, std::integral_constant<int, base + i>{}, im ? z[k] : x[m & 1][k],
                         y[m & 1][i % q]);
                });
                __builtin_amdgcn_sched_barrier(0);
            });
            put_order(std::integral_constant<int, P>{});

            // 3. back rotations and phases; the first entries of the next half are on their way
            auto accumulate = [&](auto nc) {
                constexpr int n = IDX(nc);
                unrolled<h, n + 1>([&](auto mc) {
                    constexpr int m = IDX(mc);
                    const float w = y[n & 1][(m - h) / 4][(m - h) % 4];
                    if constexpr (m == 0) {
                        U[tri(n)] += w;
                        asm volatile("" : "+v"(U[tri(n)]));
                    } else {
                        float &A = U[tri(n) + m], &B = V[tri(n - 1) + m - 1];
                        A = fmaf(h ? -tp[m] : cp[m], w, A);
                        B = fmaf(h ? cp[m] : tp[m], w, B);
                        // computed here: sunk to the end of the group, the products would stay live
                        asm volatile("" : "+v"(A), "+v"(B));
                    }
                });
            };
            if constexpr (h == 0) U[0] += X[0];
            get_rows(std::integral_constant<int, 1>{});
            if constexpr (h == 1) so = 32 * (uint32_t)src + ri;
            unrolled<0, GA>(gather_load);
            __builtin_amdgcn_sched_barrier(0);
            unrolled<1, P + 1>([&](auto nc) {
                constexpr int n = IDX(nc);
                if constexpr (n < P) get_rows(std::integral_constant<int, n + 1>{});
                rotate(std::integral_constant<int, 2>{}, nc, x[n & 1]);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (n > 1) accumulate(std::integral_constant<int, n - 1>{});
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (h == 1) operators(cls);
            unrolled<0, kFragAhead>([&](auto bc) { frag_load(std::integral_constant<int, 1 - h>{}, bc); });
            accumulate(std::integral_constant<int, P>{});
        });
    }

    store_item<P>(a, item, U, V);
}

__host__ __device__ constexpr int lds_bytes(int P) { return wave32_wpe(P) == 1 ? joint_lds_bytes(P) : 256 * tri(P + 1); }

// The parts of the blocks that were split over items, added in FP64 in a fixed order.  A workgroup
// takes 256 / J of a block's values (entry of U, target, part), with J threads a value: thread j adds
// the parts s = j mod J, and the J sums are added through LDS.  J = 8 for few values, which are bound
// by latency, 1 for those that fill the chip (bound by memory: 1.2 TB/s with J = 8, 2.5 with 1).
constexpr int kSumThreads = 256;
constexpr int sum_slices(int64_t values) { return values < 200000 ? 8 : 1; }

template <int J>
__device__ __forceinline__ void wave32_sum(const M2LWaveArgs& a, int P, int b, int chunk) {
    constexpr int kValues = kSumThreads / J;
    __shared__ double2 acc[J][kValues];
    const int s0 = a.part_ptr[b], n_parts = a.part_ptr[b + 1] - s0;
    const int tb2 = 2 * a.tb, NU = tri(P + 1), NV = tri(P), total = NU * tb2;
    if (n_parts == 0 || chunk * kValues >= total) return;
    const int e = threadIdx.x % kValues, j = threadIdx.x / kValues;
    const int t = min(chunk * kValues + e, total - 1), i = t / tb2, l = t % tb2;
    int n = (int)((sqrtf(8.0f * (float)i + 1.0f) - 1.0f) * 0.5f);   // the largest with tri(n) <= i
    if (tri(n + 1) <= i) ++n;
    if (tri(n) > i) --n;
    const int m = i - tri(n);
    const size_t step = (size_t)(NU + NV) * tb2;
    const float* pu = (const float*)a.part + s0 * step + t;
    const float* pv = (const float*)a.part + s0 * step + (size_t)(NU + (m ? tri(n - 1) + m - 1 : 0)) * tb2 + l;
    double u = 0.0, v = 0.0;
    for (int s = j; s < n_parts; s += 4 * J) {   // four loads of each in flight
        float wu[4], wv[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const size_t o = step * min(s + k * J, n_parts - 1);
            wu[k] = pu[o];
            wv[k] = pv[o];
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (s + k * J < n_parts) {
                u += (double)wu[k];
                v += (double)wv[k];
            }
    }
    if constexpr (J > 1) {
        acc[j][e] = make_double2(u, v);
        __syncthreads();
        if (j) return;
        for (int k = 1; k < J; ++k) {
            u += acc[k][e].x;
            v += acc[k][e].y;
        }
    }
    if (chunk * kValues + e >= total) return;
    const int tbox = a.blk_targets[(size_t)b * a.tb + l / 2];
    if (tbox < 0) return;
    store_expansion((double*)(a.L + a.exp_off[tbox]) + (l & 1), n, m, u, v);
}

template <int J>
__global__ __launch_bounds__(kSumThreads) void wave32_sum_kernel(M2LWaveArgs a, int P) {
    wave32_sum<J>(a, P, blockIdx.x, blockIdx.y);
}

__global__ __launch_bounds__(kSumThreads) void wave32_sum_batch_kernel(const M2LWaveArgs* __restrict__ args,
                                                                       const int4* __restrict__ work, int P) {
    const int4 wk = work[blockIdx.x];   // (descriptor, block, chunk)
    wave32_sum<8>(args[wk.x], P, wk.y, wk.z);
}

// blocks of operator columns and pairs of entries that loads run ahead of their use
constexpr int kFragsAhead = 2;
constexpr int pairs_ahead(int p) { return p == 11 ? 3 : p == 15 ? 5 : 8; }   // 11, 15: what 256 or 512 registers leave

template <int P>
__device__ __forceinline__ void wave32_item(const M2LWaveArgs& a, const int4 item) {
    if constexpr (wave32_wpe(P) == 1)
        wave32_joint_body<P, kFragsAhead, pairs_ahead(P)>(a, item);
    else
        wave32_split_body<P, kFragsAhead, pairs_ahead(P)>(a, item);
}

// workgroup i runs on XCD i % 8, and XCD x takes the contiguous item range [x n/8, (x+1) n/8) of
// the spatially ordered list (a multiple of 8 items)
template <int P>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(wave32_wpe(P), wave32_wpe(P)))) void wave32_kernel(
    M2LWaveArgs a) {
    const int per_xcd = a.n_items / kXcds;
    wave32_item<P>(a, a.items[(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds]);
}

// batches: one launch over the items of many translations of degree P; work[i] = (descriptor, item)
template <int P>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(wave32_wpe(P), wave32_wpe(P)))) void
wave32_batch_kernel(const M2LWaveArgs* __restrict__ args, const int2* __restrict__ work, int n) {
    const int per_xcd = n / kXcds;
    const int2 wk = work[(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds];
    const M2LWaveArgs a = args[wk.x];
    wave32_item<P>(a, a.items[wk.y]);
}

void check_launch(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) fail(-3, std::string("kernel launch failed (") + what + "): " + hipGetErrorString(e));
}

// run f(kernel, batch kernel) for degree p
template <typename F>
void with_degree(int p, F&& f) {
    switch (p) {
#define C(P)                                         \
    case P:                                          \
        f(wave32_kernel<P>, wave32_batch_kernel<P>); \
        break;
        C(2) C(3) C(4) C(5) C(6) C(7) C(8) C(9) C(10) C(11) C(12) C(13) C(14) C(15)
#undef C
        default: fail(-9, "internal: degree outside the FP32 wave kernel's range");
    }
}

// Pair i of the FP32 (S, D) form of consecutive boxes' expansions ((p+1)^2 each), entries tri(n) + m: Re S,
// Im D of both, then Im S, Re D of both; a box starts at a whole pair
__device__ __forceinline__ void to_sd32(const double2* x, float4* sd, int64_t i, int P1) {
    const int te = P1 * (P1 + 1) / 2, np = (te + 1) / 2;
    const int64_t b = i / np;
    const int e0 = 2 * (int)(i - b * np);
    float4 re = make_float4(0, 0, 0, 0), im = re;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int e = e0 + j;
        if (e >= te) break;
        int nn = (int)((sqrtf(8.0f * (float)e + 1.0f) - 1.0f) * 0.5f);   // the largest with tri(nn) <= e
        if (tri(nn + 1) <= e) ++nn;
        if (tri(nn) > e) --nn;
        const int m = e - tri(nn);
        const double2* xb = x + b * P1 * P1 + nn * nn + nn;
        const double2 xp = xb[m];
        double2 s = xp, d = make_double2(0.0, 0.0);
        if (m > 0) {
            double2 xm = xb[-m];
            if (m & 1) xm = make_double2(-xm.x, -xm.y);
            s = make_double2(xp.x + xm.x, xp.y + xm.y);
            d = make_double2(xp.x - xm.x, xp.y - xm.y);
        }
        (j ? re.z : re.x) = (float)s.x;
        (j ? re.w : re.y) = (float)d.y;
        (j ? im.z : im.x) = (float)s.y;
        (j ? im.w : im.y) = (float)d.x;
    }
    sd[2 * i] = re;
    sd[2 * i + 1] = im;
}

__global__ __launch_bounds__(256) void to_sd32_kernel(const double2* x, float4* sd, int64_t n, int P1) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) to_sd32(x, sd, i, P1);
}

// work[i] = (run, chunk of kSdChunk pairs)
__global__ __launch_bounds__(256) void to_sd32_batch_kernel(const SdRun* __restrict__ runs, const int2* __restrict__ work) {
    const int2 wk = work[blockIdx.x];
    const SdRun r = runs[wk.x];
    const int64_t i0 = (int64_t)wk.y * kSdChunk, i1 = min(r.n, i0 + kSdChunk);
    for (int64_t i = i0 + threadIdx.x; i < i1; i += 256) to_sd32(r.x, (float4*)r.sd, i, r.P1);
}

}  // namespace

void launch_m2l_wave32(const M2LWaveArgs& a, int p, hipStream_t s) {
    if (a.n_items <= 0) return;
    if (!a.overwrite || a.ps != p || a.pt != p) fail(-9, "internal: the FP32 wave kernel stores M2L sums of one degree");
    with_degree(p, [&](auto* k, auto*) { hipLaunchKernelGGL(k, dim3(a.n_items), dim3(64), lds_bytes(p), s, a); });
    check_launch("m2l wave32");
    if (!a.part) return;
    const int J = sum_slices((int64_t)a.n_blocks * tri(p + 1) * 2 * a.tb), values = kSumThreads / J;
    const dim3 grid(a.n_blocks, (tri(p + 1) * 2 * a.tb + values - 1) / values);
    hipLaunchKernelGGL(J == 1 ? wave32_sum_kernel<1> : wave32_sum_kernel<8>, grid, dim3(kSumThreads), 0, s, a, p);
    check_launch("m2l wave32 sum");
}

int wave32_sum_chunks(int p, int tb) { return (tri(p + 1) * 2 * tb + kSumThreads / 8 - 1) / (kSumThreads / 8); }

void launch_m2l_wave32_batch(const M2LWaveArgs* d_args, const int2* work, int n, const int4* sums, int n_sums, int p,
                             hipStream_t s) {
    if (n <= 0) return;
    with_degree(p, [&](auto*, auto* k) { hipLaunchKernelGGL(k, dim3(n), dim3(64), lds_bytes(p), s, d_args, work, n); });
    check_launch("m2l wave32 batch");
    if (n_sums <= 0) return;
    hipLaunchKernelGGL(wave32_sum_batch_kernel, dim3(n_sums), dim3(kSumThreads), 0, s, d_args, sums, p);
    check_launch("m2l wave32 batch sum");
}

void launch_to_sd32(const double2* x, float4* sd, int64_t n_boxes, int p, hipStream_t s) {
    const int64_t n = n_boxes * (((p + 1) * (p + 2) / 2 + 1) / 2);
    if (n <= 0) return;
    hipLaunchKernelGGL(to_sd32_kernel, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 65536)), dim3(256), 0, s, x, sd,
                       n, p + 1);
    check_launch("to_sd32");
}

void launch_to_sd32_batch(const SdRun* runs, const int2* work, int n, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(to_sd32_batch_kernel, dim3(n), dim3(256), 0, s, runs, work);
    check_launch("to_sd32 batch");
}

}  // namespace hfmm
