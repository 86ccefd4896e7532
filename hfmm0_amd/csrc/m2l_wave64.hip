// M2L, M2M and L2L in FP64 on matrix cores, one wave per work item.
//
// Expansions are carried in the basis of the reflection x_m -> (-1)^m x_{-m}, which commutes
// with every rotation about y: S_m = x_m + (-1)^m x_{-m}, D_m = x_m - (-1)^m x_{-m}, m >= 0
// (D_0 = 0).  There a rotation E_n splits into an (n+1) x (n+1) block on the S ("u") half and an
// n x n block on the D ("v") half, and the coaxial operator of order m acts on both alike.
//
// A wave holds 16 pairs (target box, source box) at a time whose displacements share the polar
// angle theta and the length |d|, hence the rotation and the coaxial operator: a group.  Pair c
// belongs to target c mod TB of the wave's block of TB targets (up to 16); a target takes up to
// 16 / TB of its own displacements per group, each with its own azimuth.  Per group and half:
//   0. gather: the source's (S, D) entries times e^{i m phi} -> u or v rows in LDS;
//   1. forward rotation per degree n, 2. coaxial operator per order m, 3. back rotation per
//      degree; stages 1 and 2 in place in LDS;
//   4. the results of 3 times e^{-i m phi}, added to the U and V accumulators in registers.
// Every product is a chain of 16 x 16 x 4 MFMAs whose 16 columns are the pairs, once for the real
// and once for the imaginary parts, so that an operator fragment feeds two MFMAs and the complex
// products need no exchange between lanes.  No other wave touches the wave's columns: there are no
// barriers, and the whole group is straight-line code for a degree P known at compile time, whose
// operator loads run ahead of their use.  Degrees above 7 take more than 256 registers, so that one
// wave per SIMD is left, and its latencies are exposed: of 584136 pairs at p = 14 (1.9 ms) the matrix
// pipe is busy 34% of the time (two thirds of that on entries of the operators, the rest on tile
// padding), other VALU instructions take 7%, and the wave waits on dependencies for a third.
// Against the block kernel's 8 targets x 1 direction per workgroup: 584136 pairs at p = 14 1.95 ms
// against 2.41, 53352 pairs at p = 10 0.13 + 0.01 ms against 0.29, the levels of 60k points on
// surfaces (p = 12) 0.99 ms against 2.00, a batch of 16 problems of 2k to 20k points (p = 10) 1.4 ms
// against 9.7.  (plan.cpp has the sizes and degrees at which a level takes this kernel.)  Where levels
// are irregular the gain is in the packing: pairs of a target fill the columns whatever their azimuth,
// where the block kernel leaves a column empty for every target without a source in the block's
// direction.
//
// Source and target degrees may differ (M2M, L2L): P is the larger, the tables are padded with
// zeros, absent source degrees enter as zeros and absent target degrees are not stored.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "kernels.h"

namespace hfmm {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) int* ScalarInts;   // uniform loads: scalar cache

__host__ __device__ constexpr int tri(int n) { return n * (n + 1) / 2; }

__device__ __forceinline__ d4 mma(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// f(std::integral_constant<int, i>) for i = A .. B - 1: indices of the register arrays are
// constants whatever the optimiser's unrolling limits
template <int A, int B, typename F>
__device__ __forceinline__ void unrolled(F&& f) {
    if constexpr (A < B) {
        f(std::integral_constant<int, A>{});
        unrolled<A + 1, B>(f);
    }
}
#define IDX(x) decltype(x)::value

// registers (4 rows) of degrees below n, and the degree of register i
constexpr int regs_before(int n) {
    int k = 0;
    for (int j = 0; j < n; ++j) k += j / 4 + 1;
    return k;
}
constexpr int reg_degree(int i) {
    int n = 0;
    while (regs_before(n + 1) <= i) ++n;
    return n;
}

// Rows of the LDS columns pass between the lane groups (the v half is read one row up from where it
// was gathered, the coaxial operators read along the degrees): LDS accesses before stay before those
// after.  A wave's LDS instructions are executed in order, so this holds the compiler only; without it
// addresses a constant apart look independent, being those of one lane.
__device__ __forceinline__ void lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
}

// U and V (v: U_re, U_im, V_re, V_im) of degree n and order m, back in the x basis: x_0 = U_0,
// x_m = (U + V) / 2, x_{-m} = (-1)^m (U - V) / 2
__device__ __forceinline__ void store_expansion(double2* dst, int n, int m, int pt, int overwrite, double4 v) {
    if (n > pt || m > n) return;
    double2* yp = dst + n * n + n + m;
    double2* ym = dst + n * n + n - m;
    const double sg = (m & 1) ? -0.5 : 0.5;
    double2 xp = m == 0 ? make_double2(v.x, v.y) : make_double2(0.5 * (v.x + v.z), 0.5 * (v.y + v.w));
    double2 xm = make_double2(sg * (v.x - v.z), sg * (v.y - v.w));
    if (!overwrite) {
        xp = make_double2(yp->x + xp.x, yp->y + xp.y);
        if (m > 0) xm = make_double2(ym->x + xm.x, ym->y + xm.y);
    }
    *yp = xp;
    if (m > 0) *ym = xm;
}

// 16 bytes at a uniform base plus a 32-bit lane offset: a scalar base register pair and one
// vector register (64-bit lane addresses of the many fragments would take the registers)
__device__ __forceinline__ double2 load16(const void* base, uint32_t off) {
    return *(const double2*)((const char*)base + off);
}

// One work item (block, first group, end group, part) at degree P: part 0 stores its sums, part
// s > 0 leaves them in slot s - 1 of the partial sums.
template <int P, int kFragAhead, int kGatherAhead>
__device__ __forceinline__ void wave64_body(const M2LWaveArgs& a, const int4 item) {
    // row tri(n) + m: 16 pairs of (re, im); the last rows pad the reads of the last block
    extern __shared__ double2 X[];
    constexpr int KP = P / 4 + 1;   // 4-row registers of a column of P + 1 rows
    const int lane = threadIdx.x, li = lane & 15, lk = lane >> 4;
    if (item.y >= item.z) return;   // padding item
    const int ps = a.ps, pt = a.pt;
    // accumulators, [register of (degree n, orders 4 r + lk)][re, im]; scalars, since vectors of
    // four would reserve registers for the orders above n
    constexpr int NR = regs_before(P + 1);
    double U[NR][2], V[NR][2];
    unrolled<0, NR>([&](auto ic) { U[IDX(ic)][0] = U[IDX(ic)][1] = V[IDX(ic)][0] = V[IDX(ic)][1] = 0.0; });
    double2* dump = X + 16 * (tri(P + 1) + 3) + lane;   // results of rows outside a block
    for (int i = lane; i < 16 * (tri(P + 1) + 3); i += 64) X[i] = make_double2(0.0, 0.0);
    lds_order();
    // LDS addresses: rows of one degree are consecutive (lane group lk: row 4 j + lk); rows of one
    // order m lie at tri(n) + m, n = 4 j + lk (degrees above P: the row of degree P, whose
    // products meet zeros of the operator)
    double2* xr = X + 16 * lk + li;
    double2* xc[KP];
#pragma unroll
    for (int j = 0; j < KP; ++j) xc[j] = X + 16 * tri(min(4 * j + lk, P)) + li;

    int src = a.grp_src[(size_t)item.y * 16 + li];
    int dir = a.grp_dir[(size_t)item.y * 16 + li];
#pragma unroll 1
    for (int e = item.y; e < item.z; ++e) {
        const int cls = ((ScalarInts)a.grp_class)[e];   // theta | dist << 16
        const double2* R1 = (const double2*)((const double*)a.rot1 + (size_t)(cls & 0xFFFF) * a.rot_stride);
        const double2* R3 = (const double2*)((const double*)a.rot3 + (size_t)(cls & 0xFFFF) * a.rot_stride);
        const double2* T = (const double2*)((const double*)a.coax + (size_t)(cls >> 16) * a.coax_stride);
        const uint32_t lane16 = 16 * (uint32_t)lane;
        // (S, D) entries of the source; degrees above the source's read the block of zeros
        const uint32_t so = 32 * (uint32_t)(src + lk), sz = 32 * (uint32_t)lk;
        double2 ph[KP];   // (cos, sin) of order 4 r + lk
#pragma unroll
        for (int r = 0; r < KP; ++r) ph[r] = ((const double2*)a.phase)[(size_t)dir * a.phase_stride + min(4 * r + lk, a.phase_stride - 1)];
        // the next group's sources and directions are on their way while this one is processed
        const int en = e + 1 < item.z ? e + 1 : e;
        src = a.grp_src[(size_t)en * 16 + li];
        dir = a.grp_dir[(size_t)en * 16 + li];

        unrolled<0, 2>([&](auto hc) {
            constexpr int h = IDX(hc);
            // 0. u = c S + i s D (h = 0), v = c D + i s S (h = 1), degrees in ascending order:
            // what a degree's last register writes past its rows the next degree overwrites.
            // kAhead registers' entries are in flight
            constexpr int kAhead = NR < kGatherAhead ? NR : kGatherAhead;
            lds_order();
            double4 g[kAhead];
            auto gather_load = [&](auto ic) {
                constexpr int i = IDX(ic), n = reg_degree(i), r = i - regs_before(n);
                const double2* m0 = (const double2*)a.M + 2 * (tri(n) + 4 * r);
                // lanes past degree P's last order read zeros too: the MFMAs of degree P read the rows
                // that they write, and 0 x NaN of an entry that this call has not written is NaN
                uint32_t o = n <= ps ? so : sz;
                if constexpr (n == P && 4 * r + 3 > P) o = 4 * r + lk <= P ? o : sz;
                const double2 s0 = load16(m0, o), d0 = load16(m0 + 1, o);
                g[i % kAhead] = make_double4(s0.x, s0.y, d0.x, d0.y);
            };
            unrolled<0, kAhead>(gather_load);
            unrolled<0, NR>([&](auto ic) {
                constexpr int i = IDX(ic), n = reg_degree(i), r = i - regs_before(n);
                const double4 s = g[i % kAhead];   // S_re, S_im, D_re, D_im
                if constexpr (i + kAhead < NR) gather_load(std::integral_constant<int, i + kAhead>{});
                const double2 o = h ? make_double2(s.z, s.w) : make_double2(s.x, s.y);
                const double2 q = h ? make_double2(s.x, s.y) : make_double2(s.z, s.w);
                xr[16 * (tri(n) + 4 * r)] = make_double2(fma(ph[r].x, o.x, -ph[r].y * q.y),
                                                         fma(ph[r].x, o.y, ph[r].y * q.x));
                if constexpr (r == n / 4 && (n % 4 != 3 || n == P)) lds_order();   // past its rows; all rows done
                __builtin_amdgcn_sched_barrier(0);
            });
            // The stages' blocks are one sequence q: forward rotations (degree h + q), coaxial
            // operators, back rotations.  Operator fragments are loaded kFragAhead blocks ahead, the
            // rows of the next block of a stage before the current one's results are stored
            // (they are other rows), so that cache and LDS latencies pass behind the products.
            constexpr int NB = P + 1 - h;   // blocks per stage
            double2 f[kFragAhead + 1][4], b[2][4];
            auto frag_load = [&](auto qc) {
                constexpr int q = IDX(qc), st = q / NB, i = h + q % NB;
                double2* ff = f[q % (kFragAhead + 1)];
                if constexpr (st == 1) {
#pragma unroll
                    for (int j = i / 4; j < KP; ++j) ff[j - i / 4] = load16(T + 64 * (wave64_coax_regs(P, i) + j - i / 4), lane16);
                } else {
                    constexpr int ks = (i + 4 - h) / 4;   // ceil((i + 1 - h) / 4)
#pragma unroll
                    for (int j = 0; j < (ks + 1) / 2; ++j) ff[j] = load16((st ? R3 : R1) + 64 * (wave64_rot_regs(i, h) + j), lane16);
                }
            };
            auto row_load = [&](auto qc) {
                constexpr int q = IDX(qc), st = q / NB, i = h + q % NB;
                double2* bb = b[q & 1];
                if constexpr (st == 1) {
#pragma unroll
                    for (int j = i / 4; j < KP; ++j) bb[j] = xc[j][16 * i];
                } else {
                    constexpr int ks = (i + 4 - h) / 4;
#pragma unroll
                    for (int j = 0; j < ks; ++j) bb[j] = xr[16 * (tri(i) + h + 4 * j)];
                }
            };
            unrolled<0, kFragAhead>([&](auto qc) {
                if constexpr (IDX(qc) < 3 * NB) frag_load(qc);
            });
            __builtin_amdgcn_sched_barrier(0);
            d4 re[2], im[2];
            // the results of a block: stored to its rows (stages 1 and 2), or times e^{-i m phi}
            // into the accumulators
            auto finish = [&](auto qc) {
                constexpr int q = IDX(qc), st = q / NB, i = h + q % NB;
                const d4 &yr = re[q & 1], &yi = im[q & 1];
                if constexpr (st == 0) {
                    constexpr int len = i + 1 - h, ks = (len + 3) / 4;
#pragma unroll
                    for (int r = 0; r < ks; ++r) {
                        double2* w = xr + 16 * (tri(i) + h + 4 * r);
                        if (4 * r + 3 >= len) w = lk < len - 4 * r ? w : dump;
                        *w = make_double2(yr[r], yi[r]);
                    }
                } else if constexpr (st == 1) {
#pragma unroll
                    for (int j = i / 4; j < KP; ++j) {
                        double2* w = xc[j] + 16 * i;
                        if (4 * j < i) w = 4 * j + lk >= i ? w : dump;
                        if (4 * j + 3 > P) w = 4 * j + lk <= P ? w : dump;
                        *w = make_double2(yr[j], yi[j]);
                    }
                } else {
                    // U += c u', V += -i s u' (h = 0); V += c v', U += -i s v' (h = 1); output row of
                    // the fragment is the order in both halves (the v half's row 0 is zero)
                    unrolled<0, i / 4 + 1>([&](auto rc) {
                        constexpr int r = IDX(rc), k = regs_before(i) + r;
                        const double c = ph[r].x, s = ph[r].y;
                        double* A = h ? V[k] : U[k];
                        double* B = h ? U[k] : V[k];
                        A[0] = fma(c, yr[r], A[0]);
                        A[1] = fma(c, yi[r], A[1]);
                        B[0] = fma(s, yi[r], B[0]);
                        B[1] = fma(-s, yr[r], B[1]);
                        // computed here: sunk to the end of the group, the products would stay live
                        asm volatile("" : "+v"(A[0]), "+v"(A[1]), "+v"(B[0]), "+v"(B[1]));
                    });
                }
            };
            unrolled<0, 3 * NB>([&](auto qc) {
                constexpr int q = IDX(qc), st = q / NB, i = h + q % NB;
                if constexpr (q % NB == 0) row_load(qc);
                if constexpr (q + kFragAhead < 3 * NB) frag_load(std::integral_constant<int, q + kFragAhead>{});
                if constexpr (q % NB < NB - 1) row_load(std::integral_constant<int, q + 1>{});
                const double2 *ff = f[q % (kFragAhead + 1)], *bb = b[q & 1];
                d4 yr{0, 0, 0, 0}, yi{0, 0, 0, 0};
                if constexpr (st == 1) {   // coaxial operator of order i on degrees i .. P: Re, Im of T
#pragma unroll
                    for (int j = i / 4; j < KP; ++j) {
                        const double2 w = ff[j - i / 4];
                        yr = mma(w.x, bb[j].x, yr);
                        yi = mma(w.x, bb[j].y, yi);
                        yr = mma(-w.y, bb[j].y, yr);
                        yi = mma(w.y, bb[j].x, yi);
                    }
                } else {                   // rotation of degree i, rows h .. i
                    constexpr int ks = (i + 4 - h) / 4;
#pragma unroll
                    for (int j = 0; j < ks; ++j) {
                        const double w = (j & 1) ? ff[j / 2].y : ff[j / 2].x;
                        yr = mma(w, bb[j].x, yr);
                        yi = mma(w, bb[j].y, yi);
                    }
                }
                re[q & 1] = yr;
                im[q & 1] = yi;
                __builtin_amdgcn_sched_barrier(0);
                // the previous block's results are taken while this one's products run
                if constexpr (q % NB > 0) finish(std::integral_constant<int, q - 1>{});
                if constexpr (q % NB == NB - 1) {
                    finish(qc);
                    lds_order();
                }
                // the loads stay the stated number of blocks ahead: moved further up they would
                // not fit the registers
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    }

    // the columns of a target (pairs c = target mod tb) added, then stored
    const int tb = a.tb;
    const int tbox = a.blk_targets[(size_t)item.x * tb + (li & (tb - 1))];
    unrolled<0, NR>([&](auto ic) {
        constexpr int k = IDX(ic), n = reg_degree(k), r = k - regs_before(n);
        double4 v = make_double4(U[k][0], U[k][1], V[k][0], V[k][1]);
        for (int off = tb; off < 16; off <<= 1) {
            v.x += __shfl_xor(v.x, off);
            v.y += __shfl_xor(v.y, off);
            v.z += __shfl_xor(v.z, off);
            v.w += __shfl_xor(v.w, off);
        }
        if (item.w > 0) {   // one of several parts of the block: summed by wave64_sum_kernel
            if (li < tb) ((double4*)a.part)[((size_t)(item.w - 1) * NR + k) * (4 * tb) + tb * lk + li] = v;
        } else if (tbox >= 0 && li < tb) {
            store_expansion(a.L + a.exp_off[tbox], n, 4 * r + lk, pt, a.overwrite, v);
        }
    });
}

// The parts of the blocks that were split over items, added in a fixed order.  A workgroup takes 32
// of the 4 tb NR values of a block (register k, order group and target), with 8 threads a value:
// thread j adds the parts s = j mod 8, and the 8 sums are added through LDS.  Bound by latency (the
// few blocks of a coarse level have up to ~190 parts): 12.5 us at 640 points and p = 6 with one
// thread a value, 5.7 with 8; 13.4 and 6.2 us on 64 targets at p = 10.
constexpr int kSumThreads = 256, kSumSlices = 8, kSumValues = kSumThreads / kSumSlices;

__device__ __forceinline__ void wave64_sum(const M2LWaveArgs& a, int P, int b, int chunk) {
    __shared__ double4 acc[kSumSlices][kSumValues];
    const int s0 = a.part_ptr[b], s1 = a.part_ptr[b + 1];
    if (s0 == s1) return;
    const int tb = a.tb, NR = regs_before(P + 1), total = NR * 4 * tb;
    const int e = threadIdx.x % kSumValues, j = threadIdx.x / kSumValues;
    const int t = min(chunk * kSumValues + e, total - 1), q = t % (4 * tb);
    const double4* p = (const double4*)a.part + (size_t)s0 * total + t;
    double4 v = make_double4(0.0, 0.0, 0.0, 0.0);
    const int n_parts = s1 - s0;
    for (int s = j; s < n_parts; s += 4 * kSumSlices) {   // four loads in flight
        double4 w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = p[(size_t)total * min(s + i * kSumSlices, n_parts - 1)];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (s + i * kSumSlices < n_parts) {
                v.x += w[i].x;
                v.y += w[i].y;
                v.z += w[i].z;
                v.w += w[i].w;
            }
    }
    acc[j][e] = v;
    __syncthreads();
    if (j || chunk * kSumValues + e >= total) return;
    for (int i = 1; i < kSumSlices; ++i) {
        v.x += acc[i][e].x;
        v.y += acc[i][e].y;
        v.z += acc[i][e].z;
        v.w += acc[i][e].w;
    }
    const int tbox = a.blk_targets[(size_t)b * tb + q % tb];
    if (tbox < 0) return;
    const int k = t / (4 * tb);
    int n = 0, k0 = 0;
    while (k0 + n / 4 + 1 <= k) k0 += n++ / 4 + 1;
    store_expansion(a.L + a.exp_off[tbox], n, 4 * (k - k0) + q / tb, a.pt, a.overwrite, v);
}

__global__ __launch_bounds__(kSumThreads) void wave64_sum_kernel(M2LWaveArgs a, int P) {
    wave64_sum(a, P, blockIdx.x, blockIdx.y);
}

__global__ __launch_bounds__(kSumThreads) void wave64_sum_batch_kernel(const M2LWaveArgs* __restrict__ args,
                                                                       const int4* __restrict__ work, int P) {
    const int4 wk = work[blockIdx.x];   // (descriptor, block, chunk)
    wave64_sum(args[wk.x], P, wk.y, wk.z);
}

// Waves per SIMD: two while the accumulators leave room in 256 registers (held to 256, p = 8 spills
// 40 registers and p = 10 260).
__host__ __device__ constexpr int wave64_wpe(int p) { return p <= 7 ? 2 : 1; }
// blocks and registers that loads run ahead of their use
__host__ __device__ constexpr int wave64_frag_ahead(int p) { return p <= 7 ? 2 : p <= 11 ? 4 : p <= 13 ? 2 : 1; }
__host__ __device__ constexpr int wave64_gather_ahead(int p) { return p <= 7 ? 8 : p <= 11 ? 16 : p <= 12 ? 10 : p <= 13 ? 8 : 4; }

// one launch per translation; workgroup i runs on XCD i % 8, and XCD x takes the contiguous
// item range [x n/8, (x+1) n/8) of the spatially ordered list (a multiple of 8 items)
template <int P>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(wave64_wpe(P), wave64_wpe(P)))) void wave64_kernel(
    M2LWaveArgs a) {
    const int per_xcd = a.n_items / kXcds;
    wave64_body<P, wave64_frag_ahead(P), wave64_gather_ahead(P)>(a, a.items[(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds]);
}

// batches: one launch over the items of many translations of degree P; work[i] = (descriptor, item)
template <int P>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(wave64_wpe(P), wave64_wpe(P)))) void
wave64_batch_kernel(const M2LWaveArgs* __restrict__ args, const int2* __restrict__ work, int n) {
    const int per_xcd = n / kXcds;
    const int2 wk = work[(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds];
    const M2LWaveArgs a = args[wk.x];
    wave64_body<P, wave64_frag_ahead(P), wave64_gather_ahead(P)>(a, a.items[wk.y]);
}

void check_launch(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) fail(-3, std::string("kernel launch failed (") + what + "): " + hipGetErrorString(e));
}

// run f(kernel, batch kernel) for degree p
template <typename F>
void with_degree(int p, F&& f) {
    switch (p) {
#define C(P)                                                \
    case P:                                                 \
        f(wave64_kernel<P>, wave64_batch_kernel<P>); \
        break;
        C(2) C(3) C(4) C(5) C(6) C(7) C(8) C(9) C(10) C(11) C(12) C(13) C(14)
#undef C
        default: fail(-9, "internal: degree outside the FP64 wave kernel's range");
    }
}

// Entry i of the (S, D) form (S_re, S_im, D_re, D_im; tri(n) + m within a box) of consecutive boxes'
// expansions ((p+1)^2 each)
__device__ __forceinline__ void to_sd64(const double2* x, double4* sd, int64_t i, int P1) {
    const int te = P1 * (P1 + 1) / 2;
    const int64_t b = i / te;
    const int e = (int)(i - b * te);
    int nn = (int)((sqrtf(8.0f * (float)e + 1.0f) - 1.0f) * 0.5f);   // the largest with tri(nn) <= e
    if (tri(nn + 1) <= e) ++nn;
    if (tri(nn) > e) --nn;
    const int m = e - tri(nn);
    const double2* xb = x + b * P1 * P1 + nn * nn + nn;
    const double2 xp = xb[m];
    double4 o = make_double4(xp.x, xp.y, 0.0, 0.0);
    if (m > 0) {
        double2 xm = xb[-m];
        if (m & 1) xm = make_double2(-xm.x, -xm.y);
        o = make_double4(xp.x + xm.x, xp.y + xm.y, xp.x - xm.x, xp.y - xm.y);
    }
    sd[i] = o;
}

__global__ __launch_bounds__(256) void to_sd64_kernel(const double2* x, double4* sd, int64_t n, int P1) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) to_sd64(x, sd, i, P1);
}

// work[i] = (run, chunk of kSdChunk entries)
__global__ __launch_bounds__(256) void to_sd64_batch_kernel(const SdRun* __restrict__ runs, const int2* __restrict__ work) {
    const int2 wk = work[blockIdx.x];
    const SdRun r = runs[wk.x];
    const int64_t i0 = (int64_t)wk.y * kSdChunk, i1 = min(r.n, i0 + kSdChunk);
    for (int64_t i = i0 + threadIdx.x; i < i1; i += 256) to_sd64(r.x, (double4*)r.sd, i, r.P1);
}

size_t lds_bytes(int p) { return (size_t)16 * (tri(p + 1) + 7) * sizeof(double2); }

}  // namespace

void launch_m2l_wave64(const M2LWaveArgs& a, int p, hipStream_t s) {
    if (a.n_items <= 0) return;
    with_degree(p, [&](auto* k, auto*) { hipLaunchKernelGGL(k, dim3(a.n_items), dim3(64), lds_bytes(p), s, a); });
    check_launch("m2l wave64");
    if (!a.part) return;
    hipLaunchKernelGGL(wave64_sum_kernel, dim3(a.n_blocks, wave64_sum_chunks(p, a.tb)), dim3(kSumThreads), 0, s, a, p);
    check_launch("m2l wave64 sum");
}

int wave64_sum_chunks(int p, int tb) { return (regs_before(p + 1) * 4 * tb + kSumValues - 1) / kSumValues; }

void launch_m2l_wave64_batch(const M2LWaveArgs* d_args, const int2* work, int n, const int4* sums, int n_sums, int p,
                             hipStream_t s) {
    if (n <= 0) return;
    with_degree(p, [&](auto*, auto* k) { hipLaunchKernelGGL(k, dim3(n), dim3(64), lds_bytes(p), s, d_args, work, n); });
    check_launch("m2l wave64 batch");
    if (n_sums <= 0) return;
    hipLaunchKernelGGL(wave64_sum_batch_kernel, dim3(n_sums), dim3(kSumThreads), 0, s, d_args, sums, p);
    check_launch("m2l wave64 batch sum");
}

void launch_to_sd64(const double2* x, double4* sd, int64_t n_boxes, int p, hipStream_t s) {
    const int64_t n = n_boxes * tri(p + 1);
    if (n <= 0) return;
    hipLaunchKernelGGL(to_sd64_kernel, dim3((unsigned)std::min<int64_t>((n + 255) / 256, 65536)), dim3(256), 0, s, x, sd,
                       n, p + 1);
    check_launch("to_sd64");
}

void launch_to_sd64_batch(const SdRun* runs, const int2* work, int n, hipStream_t s) {
    if (n <= 0) return;
    hipLaunchKernelGGL(to_sd64_batch_kernel, dim3(n), dim3(256), 0, s, runs, work);
    check_launch("to_sd64 batch");
}

}  // namespace hfmm
