// Plan creation (tree, lists, operator tables, device buffers), the evaluate sequence
// and the C ABI declared in include/hfmm.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstring>
#include <functional>
#include <limits>
#include <map>
#include <memory>
#include <tuple>
#include <numeric>
#include <string>
#include <vector>

#include "../../include/hfmm.h"
#include "common.h"
#include "kernels.h"
#include "p2p_math.h"

namespace hfmm {

void fail(int code, const std::string& msg) { throw Error{code, msg}; }

static thread_local std::string g_last_error;
void set_last_error(const std::string& msg) { g_last_error = msg; }

#define HIPCHK(call)                                                                              \
    do {                                                                                          \
        hipError_t e_ = (call);                                                                   \
        if (e_ != hipSuccess) fail(HFMM_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
    } while (0)

constexpr int kDirV = 0;         // 343 same-level displacements
constexpr int kDirM2M = 343;     // 8 child octants, t = c_parent - c_child
constexpr int kDirL2L = 351;     // 8 child octants, t = c_child - c_parent
constexpr int kNumDirs = 359;

inline bool real_charges(int q_type) { return q_type == HFMM_F64 || q_type == HFMM_F32; }
inline size_t charge_bytes(int q_type) {
    return q_type == HFMM_C128 ? 16 : (q_type == HFMM_F32 ? 4 : 8);
}

struct M2LBlockLevel {
    bool use = false;
    bool fp32 = false;             // kernel precision (M2L of a mixed-precision level)
    int tb = 0;                    // target boxes per workgroup
    int grp = 1;                   // directions per group
    int ps = 0, pt = 0;            // source and target table degrees
    int src_level = 0, tgt_level = 0;
    int n_items = 0;
    int4* items = nullptr;
    int* targets = nullptr;
    unsigned short* dir = nullptr;
    int* off = nullptr;
    int* units1 = nullptr;
    int n_units1 = 0;
    int* units2 = nullptr;
    int n_units2 = 0;
    int* units3 = nullptr;
    int n_units3 = 0;
    void* coax = nullptr;          // A fragments of the coaxial tables, kernel precision
    int* coax_off = nullptr;       // per order m
    int* coax_offq = nullptr;      // per order m: its 4 x 4 fragment (-1: block larger than 4 x 4)
    int coax_stride = 0;
    bool split = false;            // M2M split over items: the targets are cleared first
    int n_zero = 0;                // targets to clear
    int* zero = nullptr;
};

// L2P takes leaves of levels of different degrees in launches of their own, each with the LDS (and so
// the resident workgroups) of its degree, where every launch has this many: about the workgroups that
// fit the chip at once.  200k clustered points, degrees 13, 12 and 11 on the levels with leaves: L2P
// 0.204 ms in one launch sized for degree 13, 0.162 in three (evaluate 3.045 -> 2.995 ms).
constexpr int kL2PRunLeaves = 3072;

// items an M2L launch of the FP64 wave kernel is split into (m2l_wave64.hip)
constexpr int kWaveItems = 3072;

// Translation of one level with one wave per work item (m2l_wave64.hip, m2l_wave32.hip)
struct M2LWaveLevel {
    bool use = false;
    bool fp32 = false;
    int tb = 0;                    // targets per block
    int ps = 0, pt = 0;            // table degrees
    int src_level = 0, tgt_level = 0;
    int n_items = 0;
    int4* items = nullptr;
    int* targets = nullptr;
    int* cls = nullptr;
    int* src = nullptr;
    unsigned short* dir = nullptr;
    std::vector<double> tab;       // packed coaxial tables (host): fragments are made per degree
    int n_dist = 0;
    void* coax = nullptr;          // fragments for the effective degrees
    int coax_stride = 0;
    int n_blocks = 0, n_slots = 0;
    int* part_ptr = nullptr;
    void* part = nullptr;          // partial sums of blocks split over items, shared by the levels
    int n_groups = 0;
    std::vector<int> host_part_ptr;            // ... FP32: the slots of the plan's own split
    std::vector<int> host_targets, host_ptr;   // plans of a batch: blocks and their groups,
                                   // which the batch splits anew
};

struct XlateLaunch {
    int n_targets = 0;
    int* targets = nullptr;
    int* ptr = nullptr;
    int* src = nullptr;
    unsigned short* dir = nullptr;
    double2* coax = nullptr;
    int64_t coax_stride = 0;
    int ps = 0, pt = 0;            // table degrees of the source / target level
    int src_level = 0, tgt_level = 0;
};

}  // namespace hfmm

using namespace hfmm;

struct hfmm_plan {
    Tree tree;
    Lists lists;
    int64_t n = 0;
    double k = 0.0;                 // |k|
    int conj = 0;                   // k < 0: conjugate charges in and results out
    int precision = HFMM_PREC_FP64;
    int use_graph = 1;
    int depth = 0;
    int pmax = 0;
    int p_level[kMaxLevels] = {0};  // table degree per level (tables, storage, LDS)
    int p_eff[kMaxLevels] = {0};    // degree evaluated per level (<= p_level)
    double h[kMaxLevels] = {0}, R[kMaxLevels] = {0};
    std::vector<int64_t> exp_off;
    int64_t n_coef = 0;
    int64_t n_p2p_pairs = 0;
    int n_leaves = 0, n_far_leaves = 0, p2m_chunk = 8, p_leafmax = 2;
    int n_p2p_fp32 = 0;             // leading leaves of the FP32 near field (phase in FP32)
    bool p2p_lowk = false;          // every near pair has k r <= kP2PLowKr (mixed form)
    std::vector<double> box_maxabs; // setup only: largest |x| of the points of each box
    double* d_floor2 = nullptr;     // per leaf (leaf_box order): coincidence floor on r^2
    unsigned degree_version = 0;    // bumped by set_degrees (graphs that captured this plan are stale)

    std::vector<void*> allocs;
    double *dX = nullptr, *dY = nullptr, *dZ = nullptr;
    int* d_perm = nullptr;
    double* d_centre = nullptr;
    int *d_level = nullptr, *d_pstart = nullptr, *d_count = nullptr;
    int64_t* d_expoff = nullptr;
    int* d_plevel = nullptr;
    double* d_R = nullptr;
    int* d_far_leaves = nullptr;
    LeafDesc* d_leafdesc = nullptr;   // per far leaf (d_far_leaves order): P2M / L2P descriptors
    struct LeafRun { int first, n, p; };
    std::vector<LeafRun> l2p_runs;    // far leaves of consecutive levels and their largest table degree
    int *d_leaf_box = nullptr, *d_batch_ptr = nullptr, *d_rng_delta = nullptr, *d_leaf_src_total = nullptr;
    NearBatch* d_batches = nullptr;
    NearItems near_items[2], field_items[2];   // FP32-phase (or FP64) leaves, FP64-phase leaves
    std::vector<int> leaf_box, leaf_total;     // plans of a batch: box and sources of each
                                               // leaf, whose items the batch makes anew
    double* d_rot = nullptr;
    double2* d_phase = nullptr;
    DispInfo* d_dinfo = nullptr;
    XlateLaunch m2l[kMaxLevels], m2m[kMaxLevels], l2l[kMaxLevels];
    M2LBlockLevel m2lb[kMaxLevels];
    bool m2l_fp32[kMaxLevels] = {};  // M2L of the level in FP32 (mixed precision)
    M2LBlockLevel m2mb[kMaxLevels], l2lb[kMaxLevels];   // M2M / L2L on matrix cores
    M2LWaveLevel m2lc[kMaxLevels], m2mc[kMaxLevels], l2lc[kMaxLevels];   // one wave per item
    bool in_batch = false;           // one of a batch (also evaluated alone)
    std::vector<int64_t> sd_off;     // offset of each box's (S, D) entries
    int64_t n_sd = 0;
    double *d_cr1 = nullptr, *d_cr3 = nullptr;   // rotation fragments of the wave kernel
    int cr_stride = 0;
    float *d_wr1 = nullptr, *d_wr3 = nullptr;    // ... and of its FP32 form
    int wr_stride = 0;
    std::vector<int64_t> sd32_off;   // offset of each box's FP32 (S, D) entries, in pairs
    int64_t n_sd32 = 0;
    float4* dMs32 = nullptr;         // multipoles as FP32 (S, D) entries, two float4 per pair
    double4 *dMs = nullptr, *dLs = nullptr;      // multipoles / parents' locals in (S, D) form
    int m2l_kernel = 0;
    int p2p_tile = 2;               // targets per lane of the mixed near field
    double p2p_coord32_tol = 0.0;   // estimated error up to which a leaf takes FP32 coordinates (<= 0: none)
    unsigned char* d_coord32 = nullptr;   // per leaf: FP32 coordinate differences (mixed, FP32 phase)
    int n_leaves_coord32 = 0;
    size_t max_lds = 65536;
    // rotation blocks as MFMA A fragments (E^T for the forward, E for the back rotation)
    double *d_rf1 = nullptr, *d_rf3 = nullptr;
    float *d_rf1_32 = nullptr, *d_rf3_32 = nullptr;
    int *d_rf_off1 = nullptr, *d_rf_off3 = nullptr;
    int* d_rf_off1q = nullptr;   // forward rotation blocks of at most 4 rows: their 4 x 4 fragments
    int* d_rf_off3p = nullptr;   // packed stage-3 units: [8 n1 + n2]
    int rf_stride1 = 0, rf_stride3 = 0;
    float2* d_phase32 = nullptr;
    float2* dM32 = nullptr;
    float2* dL32 = nullptr;         // FP32 copy of the locals that FP32 L2L translations read
    double2 *dM = nullptr, *dL = nullptr, *d_q = nullptr, *d_far = nullptr;
    void* d_qin = nullptr;          // staging for host input
    double2* d_out = nullptr;       // staging for host output

    hipStream_t stream = nullptr;
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph = nullptr;
    const void* g_q = nullptr;
    void* g_out = nullptr;
    int g_qtype = -1;
    int g_outtype = -1;
    float2* d_out32 = nullptr;      // staging of complex64 output for host pointers
    double2* d_far_e = nullptr;     // far field E (sorted order), allocated at the first field call
    double2* d_field_out = nullptr; // staging of the field for host pointers

    template <typename T>
    T* alloc(size_t count) {
        if (count == 0) count = 1;
        void* p = nullptr;
        hipError_t e = hipMalloc(&p, count * sizeof(T));
        if (e != hipSuccess) fail(HFMM_ERR_MEMORY, std::string("hipMalloc failed: ") + hipGetErrorString(e));
        allocs.push_back(p);
        return (T*)p;
    }
    template <typename T>
    T* upload(const std::vector<T>& v) {
        T* p = alloc<T>(v.size());
        if (!v.empty()) HIPCHK(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
        return p;
    }
    ~hfmm_plan() {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        for (void* p : allocs) (void)hipFree(p);
        if (stream) (void)hipStreamDestroy(stream);
    }
    DevBoxes boxes() const { return DevBoxes{d_centre, d_level, d_pstart, d_count, d_expoff}; }
    DevLevels levels() const { return DevLevels{d_plevel, d_R}; }
};

namespace {

void check_device() {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n < 1) fail(HFMM_ERR_DEVICE, "no HIP device available");
    int dev = 0;
    HIPCHK(hipGetDevice(&dev));
    hipDeviceProp_t prop;
    HIPCHK(hipGetDeviceProperties(&prop, dev));
    if (std::string(prop.gcnArchName).find("gfx950") == std::string::npos)
        fail(HFMM_ERR_DEVICE, std::string("libhfmm is built for gfx950, found ") + prop.gcnArchName);
}

int octant(uint64_t code) { return (int)(code & 7); }

// Units of work of a translation from degree ps to degree pt: forward rotations of the u
// and v blocks of degrees n <= ps, coaxial orders |m| <= min, back rotations (n, row tile
// of the orders 0..n) with n <= pt.  The kernel
// deals list entry u to wave u % 4; the lists are laid out in rows of 4 so that every
// wave gets about the same number of MFMAs: units sorted by cost, each row's units given,
// largest first, to the waves with the least work so far.  Rows are padded with code 255,
// which every stage skips (a degree or order above any table).
void make_units(int ps, int pt, std::vector<int>& units1, std::vector<int>& units2, std::vector<int>& units3,
                bool pack3 = false) {
    std::vector<std::pair<int, int>> u1, u2, u3;   // (cost, code)
    for (int n = 0; n <= ps; ++n) {
        u1.push_back({m2l_tiles(n + 1) * ((n + 4) / 4), n});                   // u block
        if (n > 0) u1.push_back({m2l_tiles(n) * ((n + 3) / 4), n | (1 << 8)});  // v block
    }
    int n3 = 0;
    if (pack3) {   // degrees n1 + n2 = q share a unit (rows 0..7: n1, rows 8..15: n2)
        const int q = std::min(pt, kM2LPackMax);
        for (int n1 = 0; n1 <= q - n1; ++n1) {
            const int n2 = q - n1;
            if (n1 < n2)
                u3.push_back({(n1 + n2 + 5) / 4 + (n1 + n2 + 3) / 4 + 2, 256 | (n1 << 4) | n2});
            else
                u3.push_back({(n1 + 4) / 4 + (n1 + 3) / 4 + 2, n1});
        }
        n3 = q + 1;
    }
    for (int n = n3; n <= pt; ++n)
        for (int mt = 0; mt < m2l_tiles(n + 1); ++mt)
            u3.push_back({(n + 4) / 4 + (n + 3) / 4 + 2, n | (mt << 8)});   // + phase epilogue
    for (int m = 0; m <= std::min(ps, pt); ++m) {
        const int lens = ps + 1 - m, lent = pt + 1 - m;
        u2.push_back({(m ? 2 : 1) * m2l_tiles(lent) * ((lens + 3) / 4), m});
    }
    auto deal = [](std::vector<std::pair<int, int>> u, std::vector<int>& out) {
        std::stable_sort(u.begin(), u.end(), [](const std::pair<int, int>& a, const std::pair<int, int>& b) {
            return a.first > b.first;
        });
        while (u.size() % 4) u.push_back({0, 255});
        out.assign(u.size(), 255);
        long load[4] = {0, 0, 0, 0};
        for (size_t r = 0; r < u.size(); r += 4) {
            int order[4] = {0, 1, 2, 3};
            std::stable_sort(order, order + 4, [&](int a, int b) { return load[a] < load[b]; });
            for (int i = 0; i < 4; ++i) {
                out[r + order[i]] = u[r + i].second;
                load[order[i]] += u[r + i].first;
            }
        }
    };
    deal(u1, units1);
    deal(u2, units2);
    deal(u3, units3);
}

// Coaxial tables as A fragments: per distance, per order m = 0..min(ps, pt) the packed
// (pt+1-m) x (ps+1-m) block T[i][k] (row i: target degree m+i, column k: source degree
// m+k), padded to 16x16 tiles; per (row tile, k group, lane) eight values: Re then Im
// of j = 0..3.  coff[m] is the offset of order m within one distance.  Blocks of at most
// kM2LQuadMaxRows squared also get fragments for the 4x4x1 MFMA with its A broadcast from lanes 0..3: per
// 4-row tile t and k group g (t-major), lane l holds Re then Im of T[4t + l % 4][4g + j],
// j = 0..3; they follow the 16x16 fragments of the distance, at coffq[m] (-1 for larger
// blocks).
int coax_fragments(const std::vector<double>& tabs, int n_dist, int ps, int pt, std::vector<double>& cf,
                   std::vector<int>& coff, std::vector<int>& coffq) {
    const int mm = std::min(ps, pt);
    coff.assign(mm + 2, 0);
    for (int m = 0; m <= mm; ++m) coff[m + 1] = coff[m] + m2l_tiles(pt + 1 - m) * m2l_tiles(ps + 1 - m) * 64 * 8;
    int stride = coff[mm + 1];
    coffq.assign(mm + 1, -1);
    for (int m = 0; m <= mm; ++m)
        if (pt + 1 - m <= kM2LQuadMaxRows && ps + 1 - m <= kM2LQuadMaxRows) {
            coffq[m] = stride;
            stride += ((pt + 4 - m) / 4) * ((ps + 4 - m) / 4) * 64 * 8;
        }
    cf.assign((size_t)n_dist * stride, 0.0);
    const int csz = coax_size(pt, ps);
    for (int di = 0; di < n_dist; ++di) {
        const double* tab = &tabs[(size_t)di * csz * 2];
        double* dst = &cf[(size_t)di * stride];
        int off = 0;
        for (int m = 0; m <= mm; ++m) {
            const int lent = pt + 1 - m, lens = ps + 1 - m;
            const int nr = m2l_tiles(lent), nk = m2l_tiles(lens);
            for (int rt = 0; rt < nr; ++rt)
                for (int kg = 0; kg < nk; ++kg)
                    for (int lane = 0; lane < 64; ++lane)
                        for (int j = 0; j < 4; ++j) {
                            const int i = 16 * rt + (lane & 15), k = 16 * kg + 4 * j + (lane >> 4);
                            if (i >= lent || k >= lens) continue;
                            double* f = dst + coff[m] + ((size_t)(rt * nk + kg) * 64 + lane) * 8;
                            f[j] = tab[2 * (off + i * lens + k)];
                            f[4 + j] = tab[2 * (off + i * lens + k) + 1];
                        }
            if (coffq[m] >= 0) {
                const int nt4 = (lent + 3) / 4, nk4 = (lens + 3) / 4;
                for (int t4 = 0; t4 < nt4; ++t4)
                    for (int g4 = 0; g4 < nk4; ++g4)
                        for (int lane = 0; lane < 64; ++lane)
                            for (int j = 0; j < 4; ++j) {
                                const int i = 4 * t4 + (lane & 3), k = 4 * g4 + j;
                                if (i >= lent || k >= lens) continue;
                                double* f = dst + coffq[m] + ((size_t)(t4 * nk4 + g4) * 64 + lane) * 8;
                                f[j] = tab[2 * (off + i * lens + k)];
                                f[4 + j] = tab[2 * (off + i * lens + k) + 1];
                            }
            }
            off += lent * lens;
        }
    }
    return stride;
}

// Work items of target blocks: blocks in space order (the parent region of their first
// target, then octant), so that the kernel's XCD-aware item mapping gives each XCD a
// compact region whose source expansions stay in its L2; entry lists split when there
// are few blocks (if allowed); padded to a multiple of the XCD count with empty items.
std::vector<int4> make_items(const Tree& t, const std::vector<int>& blk_targets, const std::vector<int>& blk_ptr,
                             int tb, bool allow_split) {
    const int nblk = (int)blk_ptr.size() - 1;
    std::vector<int> border(nblk);
    for (int b = 0; b < nblk; ++b) border[b] = b;
    auto region = [&](int b) {
        const int t0 = blk_targets[(size_t)b * tb];
        return t0 < 0 ? ~0ull : t.code[t0];
    };
    std::stable_sort(border.begin(), border.end(), [&](int x, int y) {
        const uint64_t rx = region(x) >> 3, ry = region(y) >> 3;
        return rx != ry ? rx < ry : (region(x) & 7) < (region(y) & 7);
    });
    // measured at N = 1M, k = 40: 8 blocks (level 2) run best split 64 ways (0.12 ms against
    // 0.20 at 16), 64 blocks (level 3) at 16 ways (0.19 ms against 0.25 at 32)
    const int cap = nblk <= 16 ? 64 : 16;
    const int nsplit = allow_split ? std::max(1, std::min(cap, (2048 + nblk - 1) / std::max(nblk, 1))) : 1;
    std::vector<int4> items;
    for (int b : border) {
        const int e0 = blk_ptr[b], e1 = blk_ptr[b + 1];
        const int chunk = std::max(1, (e1 - e0 + nsplit - 1) / nsplit);
        for (int s = e0; s < e1; s += chunk)
            items.push_back(make_int4(b, s, std::min(e1, s + chunk), nsplit > 1 ? 1 : 0));
    }
    while (items.size() % kXcds) items.push_back(make_int4(0, 0, 0, 0));
    return items;
}

// Work items of the wave kernel: blocks in space order, each split into equal items of at most
// per_item groups; part_ptr[b] .. part_ptr[b + 1] are the partial sum slots of block b (none for
// a whole block).  Padded to a multiple of the XCD count.
std::vector<int4> wave_items(const Tree& t, const std::vector<int>& blk_targets, const std::vector<int>& blk_ptr, int tb,
                             int per_item, std::vector<int>& part_ptr) {
    const int nblk = (int)blk_ptr.size() - 1;
    std::vector<int> border(nblk);
    for (int b = 0; b < nblk; ++b) border[b] = b;
    std::stable_sort(border.begin(), border.end(), [&](int x, int y) {
        return t.code[blk_targets[(size_t)x * tb]] >> 3 < t.code[blk_targets[(size_t)y * tb]] >> 3;
    });
    auto parts = [&](int b) { return std::max(1, (blk_ptr[b + 1] - blk_ptr[b] + per_item - 1) / per_item); };
    part_ptr.assign(nblk + 1, 0);
    for (int b = 0; b < nblk; ++b) part_ptr[b + 1] = part_ptr[b] + (parts(b) > 1 ? parts(b) : 0);
    std::vector<int4> items;
    for (int b : border) {
        const int e0 = blk_ptr[b], n = blk_ptr[b + 1] - e0, np = parts(b);
        for (int i = 0; i < np; ++i)
            items.push_back(make_int4(b, e0 + (int)((int64_t)n * i / np), e0 + (int)((int64_t)n * (i + 1) / np),
                                      np > 1 ? part_ptr[b] + i + 1 : 0));
    }
    while (items.size() % kXcds) items.push_back(make_int4(0, 0, 0, 0));
    return items;
}

// Target blocks of the matrix-core M2L: boxes of level L with the same octant, TB at a
// time in Morton order; per block the displacements present (sorted by rotation and
// distance) with the source box of every target (-1 if that target lacks it).
void build_m2l_blocks(hfmm_plan& P, int L, const std::vector<int>& targets, const std::vector<int>& ptr,
                      const std::vector<int>& src, const std::vector<unsigned short>& dir,
                      const std::vector<double>& coax_d, int n_dist, const std::vector<DispInfo>& dinfo) {
    if (P.m2l_kernel == 1) return;
    const int p = P.p_level[L];
    if (p > kM2LBlockMaxP) return;   // higher degrees use the generic kernel (coarse levels only)
    const int fp32 = P.m2l_fp32[L];
    const int eb = fp32 ? 4 : 8;
    // the instantiation's stage-3 units per wave (FP32 one-tile instances pack small degrees)
    const int maxu = fp32 && m2l_tiles(p + 1) == 1 ? m2l_block_maxu_packed(p) : m2l_block_maxu(p);
    // shape of one operator application: TB target boxes x G directions (of equal theta
    // and |d|).  A requested pair count TB*G (m2l_kernel = 8, 16, 32, 64) takes the first
    // fitting shape with that count in the order below (larger TB first: partly filled
    // direction groups waste columns, target blocks rarely do).  Otherwise, from
    // measurements at N = 1M, k = 40 (finest level, 5.4M pairs): FP32 takes 16 x 2 up to
    // p = 11 (5.27 ms at p = 11 against 5.61 for 8 x 2) and 8 x 2 above (see below); FP64
    // takes 8 x 1 (38.9 ms at p = 17 against 48.4 for 8 x 2); then the next smaller shape
    // that fits.
    auto fits = [&](int c, int g) {
        if (!fp32 && !(c == 8 || (c == 16 && g == 1))) return false;   // FP64 instantiations
        if (m2l_acc_regs(maxu, c, eb) > kM2LMaxAccRegs) return false;
        return m2l_block_lds_bytes(p, c, g, eb) <= P.max_lds;
    };
    int tb = 0, grp = 0;
    const int shapes[6][2] = {{16, 4}, {16, 2}, {8, 4}, {8, 2}, {16, 1}, {8, 1}};
    if (P.m2l_kernel > 1)
        for (auto& sh : shapes)
            if (!tb && sh[0] * sh[1] == P.m2l_kernel && fits(sh[0], sh[1])) tb = sh[0], grp = sh[1];
    // with the packed stage-3 units the one-tile FP32 instances fit 16 x 2 up to p = 15:
    // at p = 12 on the finest level (32768 targets) 5.20 ms against 6.0 for 8 x 2, but on
    // the 4096 targets of level 4 0.96 against 0.80 ms (fewer, longer work items)
    const int pref[3][2][2] = {{{16, 2}, {8, 2}}, {{8, 2}, {8, 1}}, {{8, 1}, {8, 2}}};
    const bool wide = p <= 11 || (p <= 15 && targets.size() >= 16384);
    const int* pr = &pref[!fp32 ? 2 : wide ? 0 : 1][0][0];
    for (int i = 0; i < 2 && !tb; ++i)
        if (fits(pr[2 * i], pr[2 * i + 1])) tb = pr[2 * i], grp = pr[2 * i + 1];
    for (auto& sh : shapes)
        if (!tb && fits(sh[0], sh[1])) tb = sh[0], grp = sh[1];
    if (!tb) return;
    std::vector<int> units1, units2, units3;
    make_units(p, p, units1, units2, units3, fp32 && m2l_tiles(p + 1) == 1);

    const Tree& t = P.tree;
    std::vector<int> tpos(t.n_boxes(), -1);     // target ordinal in `targets`
    for (size_t i = 0; i < targets.size(); ++i) tpos[targets[i]] = (int)i;
    std::vector<int> blk_targets, blk_ptr{0}, grp_off;
    std::vector<unsigned short> grp_dir;
    for (int o = 0; o < 8; ++o) {
        std::vector<int> boxes;
        for (int b = t.level_start[L]; b < t.level_start[L + 1]; ++b)
            if ((int)(t.code[b] & 7) == o && tpos[b] >= 0) boxes.push_back(b);
        for (size_t b0 = 0; b0 < boxes.size(); b0 += tb) {
            // (theta, dist) -> direction -> sources of the TB targets
            std::map<std::pair<int, int>, std::map<int, std::vector<int>>> ents;
            for (int j = 0; j < tb; ++j) {
                const int b = b0 + j < boxes.size() ? boxes[b0 + j] : -1;
                blk_targets.push_back(b);
                if (b < 0) continue;
                const int ti = tpos[b];
                for (int e = ptr[ti]; e < ptr[ti + 1]; ++e) {
                    const int d = dir[e];
                    auto& byd = ents[std::make_pair(dinfo[d].theta, dinfo[d].dist)];
                    auto it = byd.find(d);
                    if (it == byd.end()) it = byd.emplace(d, std::vector<int>(tb, -1)).first;
                    it->second[j] = (int)P.exp_off[src[e]];
                }
            }
            for (auto& kv : ents) {
                std::vector<std::pair<int, const std::vector<int>*>> ds;
                for (auto& dv : kv.second) ds.push_back({dv.first, &dv.second});
                for (size_t g0 = 0; g0 < ds.size(); g0 += grp)
                    for (int g = 0; g < grp; ++g) {
                        const bool has = g0 + g < ds.size();
                        grp_dir.push_back(has ? (unsigned short)ds[g0 + g].first : (unsigned short)0xFFFF);
                        for (int j = 0; j < tb; ++j) grp_off.push_back(has ? (*ds[g0 + g].second)[j] : -1);
                    }
            }
            blk_ptr.push_back((int)(grp_dir.size() / grp));
        }
    }
    const std::vector<int4> items = make_items(t, blk_targets, blk_ptr, tb, true);
    M2LBlockLevel& B = P.m2lb[L];
    B.use = true;
    B.fp32 = fp32;
    B.tb = tb;
    B.grp = grp;
    B.ps = B.pt = p;
    B.src_level = B.tgt_level = L;
    B.n_items = (int)items.size();
    B.items = P.upload(items);
    B.targets = P.upload(blk_targets);
    B.dir = P.upload(grp_dir);
    B.off = P.upload(grp_off);
    B.units1 = P.upload(units1);
    B.n_units1 = (int)units1.size();
    B.units2 = P.upload(units2);
    B.n_units2 = (int)units2.size();
    B.units3 = P.upload(units3);
    B.n_units3 = (int)units3.size();
    std::vector<double> cf;
    std::vector<int> coff, coffq;
    B.coax_stride = coax_fragments(coax_d, n_dist, p, p, cf, coff, coffq);
    if (fp32) {
        std::vector<float> c32(cf.begin(), cf.end());
        B.coax = P.upload(c32);
    } else {
        B.coax = P.upload(cf);
    }
    B.coax_off = P.upload(coff);
    B.coax_offq = P.upload(coffq);
    prepare_m2l_block(p, tb, grp, fp32);
}

// targets of a block of the tree translations, each of one direction per group
constexpr int kTreeBlock = 8;

// an M2M level with fewer blocks is split: their groups go over items that add atomically
bool tree_split(int kind, size_t n_parents) { return kind == 1 && (n_parents + kTreeBlock - 1) / kTreeBlock < 512; }

// FP32 arithmetic (FP64 results) of the M2M into level L (kind 1) or the L2L out of it (kind 2): where
// the M2L of every level from 2 to L+1 runs in FP32, since the translated expansions then only
// feed FP32 translations, whose own rounding is of the same size; a chain through an FP64 M2L
// level keeps FP64.  Split M2M levels keep FP64 as well: there the FP32 form was slower (N=1M,
// k=40: 55.7 against 40.4 us for level 4 -> 3, where the level 5 -> 4 M2M took 81.9 against 113.5 us).
bool tree_fp32(const hfmm_plan& P, int L, int kind, size_t n_parents) {
    if (P.m2l_kernel == 1 || !P.d_rf1_32 || tree_split(kind, n_parents)) return false;
    for (int l = 2; l <= L + 1; ++l)
        if (!P.m2l_fp32[l] || P.p_level[l] > kM2LBlockMaxP) return false;
    return m2l_block_lds_bytes(std::max(P.p_level[L], P.p_level[L + 1]), kTreeBlock, 1, 8) <= P.max_lds;
}

// M2M (kind 1: the parents of level L from their children) and L2L (kind 2: the children
// at level L+1 from their parents) on the matrix-core block kernel, in FP32 (tree_fp32) or FP64:
// the levels that the wave kernel does not take.  Blocks of 8 targets,
// one direction per group: an M2M block runs one group per child octant present among
// its parents, every target receiving all of its children within the one work item, so
// the result is stored (no clear of the parent multipoles is needed); an L2L block holds
// 8 children of one octant and a single group (their parents' locals), added to what
// M2L left there.  tab: the coaxial table (pt+1-m) x (ps+1-m) per m of this level pair.
void build_tree_blocks(hfmm_plan& P, int L, int kind, const std::vector<double>& tab, bool fp32) {
    if (P.m2l_kernel == 1 || !P.d_rf1) return;
    const Tree& t = P.tree;
    const int ps = kind == 1 ? P.p_level[L + 1] : P.p_level[L];
    const int pt = kind == 1 ? P.p_level[L] : P.p_level[L + 1];
    const int pm = std::max(ps, pt);
    if (pm > kM2LBlockMaxP) return;
    const int tb = kTreeBlock, grp = 1;
    if (m2l_block_lds_bytes(pm, tb, grp, 8) > P.max_lds) return;
    size_t n_parents = 0;
    std::vector<int> blk_targets, blk_ptr{0}, grp_off;
    std::vector<unsigned short> grp_dir;
    if (kind == 1) {
        // parents with children, in level order, and their child per octant
        std::vector<int> parents;
        std::vector<std::array<int, 8>> child;
        for (int c = t.level_start[L + 1]; c < t.level_start[L + 2]; ++c) {
            const int par = t.parent[c];
            if (parents.empty() || parents.back() != par) {
                parents.push_back(par);
                child.push_back({-1, -1, -1, -1, -1, -1, -1, -1});
            }
            child.back()[octant(t.code[c])] = c;
        }
        n_parents = parents.size();
        for (size_t b0 = 0; b0 < parents.size(); b0 += tb) {
            for (int j = 0; j < tb; ++j) blk_targets.push_back(b0 + j < parents.size() ? parents[b0 + j] : -1);
            for (int o = 0; o < 8; ++o) {
                bool any = false;
                for (int j = 0; j < tb && b0 + j < parents.size(); ++j) any |= child[b0 + j][o] >= 0;
                if (!any) continue;
                grp_dir.push_back((unsigned short)(kDirM2M + o));
                for (int j = 0; j < tb; ++j) {
                    const int c = b0 + j < parents.size() ? child[b0 + j][o] : -1;
                    grp_off.push_back(c >= 0 ? (int)P.exp_off[c] : -1);
                }
            }
            blk_ptr.push_back((int)grp_dir.size());
        }
    } else {
        for (int o = 0; o < 8; ++o) {
            std::vector<int> kids;
            for (int c = t.level_start[L + 1]; c < t.level_start[L + 2]; ++c)
                if (octant(t.code[c]) == o) kids.push_back(c);
            for (size_t b0 = 0; b0 < kids.size(); b0 += tb) {
                grp_dir.push_back((unsigned short)(kDirL2L + o));
                for (int j = 0; j < tb; ++j) {
                    const int c = b0 + j < kids.size() ? kids[b0 + j] : -1;
                    blk_targets.push_back(c);
                    grp_off.push_back(c >= 0 ? (int)P.exp_off[t.parent[c]] : -1);
                }
                blk_ptr.push_back((int)grp_dir.size());
            }
        }
    }
    if (blk_ptr.size() < 2) return;
    // coarse M2M levels have few blocks: their groups (child octants) are split over items
    // that add atomically, after the parents are cleared; L2L blocks hold one group
    const bool split = tree_split(kind, n_parents);
    const std::vector<int4> items = make_items(t, blk_targets, blk_ptr, tb, split);
    std::vector<int> units1, units2, units3;
    make_units(ps, pt, units1, units2, units3, fp32 && m2l_tiles(pm + 1) == 1);
    M2LBlockLevel& B = kind == 1 ? P.m2mb[L] : P.l2lb[L];
    B.use = true;
    B.fp32 = fp32;
    B.tb = tb;
    B.grp = grp;
    B.ps = ps;
    B.pt = pt;
    B.src_level = kind == 1 ? L + 1 : L;
    B.tgt_level = kind == 1 ? L : L + 1;
    B.n_items = (int)items.size();
    B.items = P.upload(items);
    B.targets = P.upload(blk_targets);
    B.dir = P.upload(grp_dir);
    B.off = P.upload(grp_off);
    B.units1 = P.upload(units1);
    B.n_units1 = (int)units1.size();
    B.units2 = P.upload(units2);
    B.n_units2 = (int)units2.size();
    B.units3 = P.upload(units3);
    B.n_units3 = (int)units3.size();
    B.split = split;
    if (split) {
        std::vector<int> z;
        for (int b : blk_targets)
            if (b >= 0) z.push_back(b);
        B.n_zero = (int)z.size();
        B.zero = P.upload(z);
    }
    std::vector<double> cf;
    std::vector<int> coff, coffq;
    B.coax_stride = coax_fragments(tab, 1, ps, pt, cf, coff, coffq);
    if (fp32) {
        std::vector<float> c32(cf.begin(), cf.end());
        B.coax = P.upload(c32);
    } else {
        B.coax = P.upload(cf);
    }
    B.coax_off = P.upload(coff);
    B.coax_offq = P.upload(coffq);
    prepare_m2l_block(pm, tb, grp, fp32);
}

// Coaxial fragments of a level for its effective degrees, into B.coax
void pack_wave_coax(const hfmm_plan& P, M2LWaveLevel& B) {
    const int ps = P.p_eff[B.src_level], pt = P.p_eff[B.tgt_level], pm = std::max(ps, pt);
    if (B.fp32) {
        const int csz = coax_size(B.pt, B.ps);
        B.coax_stride = 256 * wave32_blocks(wave32_coax_vecs(pm, pm + 1));
        std::vector<float> cf((size_t)B.n_dist * B.coax_stride, 0.0f);
        for (int d = 0; d < B.n_dist; ++d) {
            size_t off = (size_t)d * csz;
            float* f = &cf[(size_t)d * B.coax_stride];
            for (int m = 0; m <= std::min(B.ps, B.pt); ++m) {
                const int lens = B.ps + 1 - m, q = (pm + 1 - m + 3) / 4;
                for (int n2 = m; n2 <= pt; ++n2)
                    for (int n = m; n <= ps; ++n) {
                        const size_t t = off + (size_t)(n2 - m) * lens + n - m;
                        const int v = wave32_coax_vecs(pm, m) + 2 * q * (n - m) + (n2 - m) / 4;
                        f[wave32_pos(v, (n2 - m) % 4)] = (float)B.tab[2 * t];
                        f[wave32_pos(v + q, (n2 - m) % 4)] = (float)B.tab[2 * t + 1];
                    }
                off += (size_t)(B.pt + 1 - m) * lens;
            }
        }
        HIPCHK(hipMemcpy(B.coax, cf.data(), cf.size() * sizeof(float), hipMemcpyHostToDevice));
        return;
    }
    const int regs = wave64_coax_regs(pm, pm + 1), csz = coax_size(B.pt, B.ps);
    B.coax_stride = regs * 128;
    std::vector<double> cf((size_t)B.n_dist * B.coax_stride, 0.0);
    for (int d = 0; d < B.n_dist; ++d) {
        size_t off = (size_t)d * csz;
        for (int m = 0; m <= std::min(B.ps, B.pt); ++m) {
            const int lens = B.ps + 1 - m;
            for (int n2 = m; n2 <= pt; ++n2)
                for (int n = m; n <= ps; ++n) {
                    const size_t t = off + (size_t)(n2 - m) * lens + n - m;
                    double* f = &cf[(size_t)d * B.coax_stride +
                                    ((size_t)(wave64_coax_regs(pm, m) + n / 4 - m / 4) * 64 + 16 * (n % 4) + n2) * 2];
                    f[0] = B.tab[2 * t];
                    f[1] = B.tab[2 * t + 1];
                }
            off += (size_t)(B.pt + 1 - m) * lens;
        }
    }
    HIPCHK(hipMemcpy(B.coax, cf.data(), cf.size() * sizeof(double), hipMemcpyHostToDevice));
}

// Pairs from which the M2L of a level runs on the wave kernels.  Below, the level is over in one wave per
// group whatever their number: the time is that of fetching the straight-line code, and of the launches
// for the sums and the (S, D) form, while the block kernel's is a few sources per target.  Whole
// evaluates with one M2L level, wave against block kernel, FP64: 190 pairs 44.3 / 41.6 us at p = 2, 59.9 / 50.9
// at p = 8, 87.5 / 63.2 at p = 14; 514 pairs 44.7 / 45.8, 61.6 / 62.3, 91.3 / 86.2; 986 pairs 44.2 / 49.0, 61.2 /
// 73.2, 99.3 / 104.9 (but a level of 956 at p = 14 10 us longer).  FP32, whose sums are shorter: 34 pairs
// 40.8 / 43.3 at p = 2, 56.2 / 56.2 at p = 10; 190 pairs 64.1 / 69.4 at p = 11, 78.1 / 69.5 at p = 14; 388
// pairs 78.1 / 84.0 at p = 14, 106 / 83.5 at p = 15.  A batch's FP64 levels share their launches and take
// the wave kernel at any size (64 problems of 30 points at p = 9: M2L 0.25 ms, 1.38 on the block kernel);
// its FP32 levels follow the plan's own rule, so that a problem's result is the one it has alone.
int wave_min_pairs(int p, bool fp32) {
    if (fp32) return p <= 10 ? 0 : p == 11 ? 128 : p <= 14 ? 288 : 960;
    return p <= 13 ? 128 + 48 * p : 1024;
}

// Largest degrees whose M2M and L2L run on the wave kernel: their few directions suit the block kernel,
// and above p = 7 the wave kernel has one wave per SIMD.  Levels 4 and 5 of 600k points, wave against block
// kernel, M2M: 0.39 / 0.57 ms at p = 7, 0.75 / 0.81 at 10, 0.86 / 0.85 at 11, 1.06 / 0.97 at 12, 1.53 / 1.09 at
// 14; L2L: 0.35 / 0.67 at p = 7, 0.82 / 1.05 at 10, 1.13 / 1.30 at 12, 1.29 / 1.40 at 13, 1.68 / 1.58 at 14.
constexpr int kWaveM2MMaxP = 10, kWaveL2LMaxP = 13;

// Translation of one level on the wave kernel: targets with their (source, direction) lists.
// kind 0: M2L, 1: M2M, 2: L2L; coax: packed tables as X.coax (interleaved complex).
void build_waves(hfmm_plan& P, M2LWaveLevel& B, int kind, int src_level, int tgt_level, const std::vector<int>& targets,
                   const std::vector<int>& ptr, const std::vector<int>& src, const std::vector<unsigned short>& dir,
                   const std::vector<double>& coax, int n_dist, const std::vector<DispInfo>& dinfo, bool fp32 = false) {
    const int ps = P.p_level[src_level], pt = P.p_level[tgt_level], pm = std::max(ps, pt);
    if (P.m2l_kernel != 0 || pm > (fp32 ? kWave32MaxP : kWave64MaxP) || !P.d_cr1) return;
    if (kind == 0 && (fp32 || !P.in_batch) && (int)src.size() < wave_min_pairs(pm, fp32)) return;
    if ((kind == 1 && pm > kWaveM2MMaxP) || (kind == 2 && pm > kWaveL2LMaxP)) return;
    // the kernels address the sources with 32-bit byte offsets
    const int64_t bytes = fp32 ? (P.n_sd32 + wave32_sd_pad(P.pmax)) * 2 * (int64_t)sizeof(float4)
                               : (P.n_sd + wave_sd_pad(P.pmax)) * (int64_t)sizeof(double4);
    if (bytes > (int64_t)UINT32_MAX) return;
    const Tree& t = P.tree;
    const int nt = (int)targets.size();
    const int pairs = fp32 ? kWave32Pairs : kWave64Pairs;
    // classes (theta, dist) present, and the targets ordered by the octant's z bit, then in
    // space: V displacements of one z bit have the same classes
    std::vector<int> cls_of(kNumDirs, -1), cls_key;
    {
        std::map<std::pair<int, int>, int> ids;
        std::vector<char> present(kNumDirs, 0);
        for (unsigned short d : dir) present[d] = 1;
        for (int d = 0; d < kNumDirs; ++d)
            if (present[d]) ids.emplace(std::make_pair(dinfo[d].theta, dinfo[d].dist), 0);
        for (auto& kv : ids) {
            kv.second = (int)cls_key.size();
            cls_key.push_back(kv.first.first | kv.first.second << 16);
        }
        for (int d = 0; d < kNumDirs; ++d) {
            auto it = ids.find(std::make_pair(dinfo[d].theta, dinfo[d].dist));
            if (it != ids.end()) cls_of[d] = it->second;
        }
    }
    const int nc = (int)cls_key.size();
    std::vector<int> order(nt);
    for (int i = 0; i < nt; ++i) order[i] = i;
    if (kind != 1)
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
            return ((t.code[targets[x]] >> 2) & 1) < ((t.code[targets[y]] >> 2) & 1);
        });
    std::vector<unsigned short> cnt((size_t)nt * nc, 0);
    for (int i = 0; i < nt; ++i)
        for (int e = ptr[i]; e < ptr[i + 1]; ++e) ++cnt[(size_t)i * nc + cls_of[dir[e]]];
    // targets per block: the one with the fewest groups (each is 16 or 32 pairs of work); on a tie the
    // smaller, whose blocks are more and end in fewer stores
    int tb = 0;
    int64_t best = 0, best_cost = 0;
    for (int c = 2; c <= pairs; c *= 2) {
        const int slots = pairs / c;
        int64_t g = 0;
        for (int b0 = 0; b0 < nt; b0 += c)
            for (int k = 0; k < nc; ++k) {
                int mx = 0;
                for (int j = b0; j < std::min(nt, b0 + c); ++j) mx = std::max<int>(mx, cnt[(size_t)order[j] * nc + k]);
                g += (mx + slots - 1) / slots;
            }
        // FP32: an item leaves c targets' sums in memory, about c / 64 of a group's time.  On 5.4M pairs
        // c = 16 and 32 both need 193.6k groups; the sums of 32 took 157 us against 65.
        const int64_t cost = g + (fp32 ? (int64_t)kWaveItems * c / 64 : 0);
        if (!tb || cost < best_cost) tb = c, best = g, best_cost = cost;
    }
    // M2M and L2L take the kernel from 2 groups per SIMD on: a launch of a group or two per wave spends
    // most of its time on fetching the code (M2M of 512 children at p = 10: 42 us, 20 on the block kernel).
    if (kind != 0 && best < 2048) return;
    const int slots = pairs / tb, nblk = (nt + tb - 1) / tb;
    std::vector<int> blk_targets((size_t)nblk * tb, -1), blk_ptr{0}, gcls, gsrc;
    std::vector<unsigned short> gdir;
    gsrc.reserve((size_t)best * pairs);
    gdir.reserve((size_t)best * pairs);
    std::vector<int> first(nc + 1), fill(nc);
    for (int b = 0; b < nblk; ++b) {
        const int j0 = b * tb, j1 = std::min(nt, j0 + tb);
        first[0] = (int)gcls.size();
        for (int k = 0; k < nc; ++k) {
            int mx = 0;
            for (int j = j0; j < j1; ++j) mx = std::max<int>(mx, cnt[(size_t)order[j] * nc + k]);
            const int g = (mx + slots - 1) / slots;
            for (int i = 0; i < g; ++i) gcls.push_back(cls_key[k]);
            first[k + 1] = first[k] + g;
        }
        gsrc.resize(gcls.size() * pairs, 0);
        gdir.resize(gcls.size() * pairs, 0);
        for (int j = j0; j < j1; ++j) {
            const int i = order[j];
            blk_targets[j] = targets[i];
            std::fill(fill.begin(), fill.end(), 0);
            for (int e = ptr[i]; e < ptr[i + 1]; ++e) {
                const int k = cls_of[dir[e]], f = fill[k]++;
                const size_t o = (size_t)(first[k] + f / slots) * pairs + (f % slots) * tb + (j - j0);
                gsrc[o] = (int)(fp32 ? P.sd32_off : P.sd_off)[src[e]];
                gdir[o] = dir[e];
            }
        }
        blk_ptr.push_back((int)gcls.size());
    }
    B.use = true;
    B.fp32 = fp32;
    B.tb = tb;
    B.ps = ps;
    B.pt = pt;
    B.src_level = src_level;
    B.tgt_level = tgt_level;
    B.targets = P.upload(blk_targets);
    B.cls = P.upload(gcls);
    B.src = P.upload(gsrc);
    B.dir = P.upload(gdir);
    B.tab = coax;
    B.n_dist = n_dist;
    B.coax = P.alloc<char>((size_t)n_dist * (fp32 ? 256 * wave32_blocks(wave32_coax_vecs(pm, pm + 1)) * sizeof(float)
                                                  : wave64_coax_regs(pm, pm + 1) * 128 * sizeof(double)));
    pack_wave_coax(P, B);
    B.n_blocks = nblk;
    B.n_groups = blk_ptr[nblk];
    // M2L blocks are split into items whose sums meet in a second kernel
    std::vector<int> part_ptr;
    int per_item = B.n_groups;
    if (kind == 0 && fp32) {
        // An item's start and end cost about half a group, and a wave too many a whole round: one
        // item for each wave that runs at a time, up to three where they keep 16 groups.  The 2900
        // items of a group or two that a fixed 3072 gave 512 targets at p = 11 took 82 us, 1024 43;
        // 4096 targets at p = 12 in 3040 items 0.32 + 0.03 ms (sums), in 960 0.315 + 0.009.
        const int slots = 1024 * wave32_wpe(pm);
        const int64_t max_items = (int64_t)slots * std::max(1, std::min(3, B.n_groups / slots / 16));
        int most = 1;
        for (int b = 0; b < nblk; ++b) most = std::max(most, blk_ptr[b + 1] - blk_ptr[b]);
        for (per_item = std::max<int>(1, B.n_groups / max_items); per_item < most; per_item += 1 + per_item / 32) {
            int64_t n = 0;
            for (int b = 0; b < nblk; ++b) n += std::max(1, (blk_ptr[b + 1] - blk_ptr[b] + per_item - 1) / per_item);
            if (n <= max_items) break;
        }
    } else if (kind == 0) {
        // three items for each wave that runs at a time (1024 SIMDs)
        per_item = std::max(1, (B.n_groups + kWaveItems - 1) / kWaveItems);
    }
    const std::vector<int4> items = wave_items(t, blk_targets, blk_ptr, tb, per_item, part_ptr);
    B.n_items = (int)items.size();
    B.items = P.upload(items);
    B.n_slots = part_ptr[nblk];
    B.part_ptr = P.upload(part_ptr);
    if (P.in_batch && kind == 0 && fp32) B.host_part_ptr = part_ptr;
    if (P.in_batch && kind == 0 && !fp32) {
        B.host_targets = std::move(blk_targets);
        B.host_ptr = std::move(blk_ptr);
    }
}

void build_tables(hfmm_plan& P) {
    const Tree& t = P.tree;
    // directions
    std::map<std::pair<int, int>, int> theta_idx;
    std::vector<double> thetas;
    std::vector<DispInfo> dinfo(kNumDirs, DispInfo{0, 0});
    std::vector<double> phis(kNumDirs, 0.0);
    std::map<int, int> dist_idx;       // |d|^2 -> index
    std::vector<int> dist_d2;
    auto theta_of = [&](int dz, int d2) {
        auto key = std::make_pair(dz, d2);
        auto it = theta_idx.find(key);
        if (it != theta_idx.end()) return it->second;
        int id = (int)thetas.size();
        thetas.push_back(std::acos(std::max(-1.0, std::min(1.0, dz / std::sqrt((double)d2)))));
        theta_idx[key] = id;
        return id;
    };
    for (int dx = -3; dx <= 3; ++dx)
        for (int dy = -3; dy <= 3; ++dy)
            for (int dz = -3; dz <= 3; ++dz) {
                const int d = (dx + 3) * 49 + (dy + 3) * 7 + (dz + 3);
                if (std::max(std::abs(dx), std::max(std::abs(dy), std::abs(dz))) < 2) continue;
                const int d2 = dx * dx + dy * dy + dz * dz;
                if (!dist_idx.count(d2)) {
                    dist_idx[d2] = (int)dist_d2.size();
                    dist_d2.push_back(d2);
                }
                dinfo[kDirV + d] = DispInfo{theta_of(dz, d2), dist_idx[d2]};
                phis[kDirV + d] = std::atan2((double)dy, (double)dx);
            }
    for (int o = 0; o < 8; ++o) {
        const int sx = 2 * (o & 1) - 1, sy = 2 * ((o >> 1) & 1) - 1, sz = 2 * ((o >> 2) & 1) - 1;
        dinfo[kDirM2M + o] = DispInfo{theta_of(-sz, 3), 0};
        phis[kDirM2M + o] = std::atan2((double)-sy, (double)-sx);
        dinfo[kDirL2L + o] = DispInfo{theta_of(sz, 3), 0};
        phis[kDirL2L + o] = std::atan2((double)sy, (double)sx);
    }
    const int pmax = P.pmax;
    const int rsz = rot_size(pmax);
    std::vector<double> rot((size_t)thetas.size() * rsz);
    for (size_t i = 0; i < thetas.size(); ++i) rotation_table(thetas[i], pmax, &rot[i * rsz]);
    P.d_rot = P.upload(rot);
    if (P.m2l_kernel != 1) {
        // rotation blocks n <= min(pmax, kM2LBlockMaxP) in the (u, v) basis as A fragments:
        // rf1 holds the blocks of E_n^T (forward rotation; u and v in their LDS order),
        // rf3 those of E_n (back rotation; output rows of both blocks indexed by the order
        // m = 0..n, the v block's row 0 zero, inputs in LDS order)
        const int pb = std::min(pmax, kM2LBlockMaxP);
        std::vector<int> off1(2 * (pb + 1), 0), off3(2 * (pb + 1), 0);
        int s1 = 0, s3 = 0;
        for (int n = 0; n <= pb; ++n) {
            off1[2 * n] = s1;
            s1 += m2l_tiles(n + 1) * m2l_tiles(n + 1) * 256;
            off1[2 * n + 1] = s1;
            s1 += m2l_tiles(n) * m2l_tiles(n) * 256;
            off3[2 * n] = s3;
            s3 += m2l_tiles(n + 1) * m2l_tiles(n + 1) * 256;
            off3[2 * n + 1] = s3;
            s3 += m2l_tiles(n + 1) * m2l_tiles(n) * 256;
        }
        // blocks of at most kM2LQuadMaxRows rows also get fragments for the 4x4x1 MFMA with its A broadcast
        // from lanes 0..3 (per 4-row tile t and k group g, t-major: lane l holds row
        // 4t + l % 4, k = 4g..4g+3), after the 16x16 fragments
        std::vector<int> off1q(2 * (pb + 1), -1);
        for (int n = 0; n <= pb; ++n)
            for (int h = 0; h < 2; ++h) {
                const int len = h ? n : n + 1;
                if (len >= 1 && len <= kM2LQuadMaxRows) {
                    off1q[2 * n + h] = s1;
                    s1 += ((len + 3) / 4) * ((len + 3) / 4) * 256;
                }
            }
        // packed stage-3 units (n1 < n2, n1 + n2 <= kM2LPackMax): a 16 x 16 block-diagonal
        // fragment each for u (rows 0..n1 and 8..8+n2; inputs n1's n1+1, then n2's n2+1) and
        // for v (same rows; inputs n1's n1, then n2's n2)
        std::vector<int> off3p(64, -1);
        for (int n1 = 0; n1 <= kM2LPackMax; ++n1)
            for (int n2 = n1 + 1; n1 + n2 <= kM2LPackMax; ++n2)
                if (n2 <= pb) {
                    off3p[8 * n1 + n2] = s3;
                    s3 += 512;
                }
        std::vector<double> f1((size_t)thetas.size() * s1, 0.0), f3((size_t)thetas.size() * s3, 0.0);
        // A fragments of an R x K matrix a(i, k) at dst
        auto put = [](double* dst, int R, int K, const std::function<double(int, int)>& a) {
            const int nk = m2l_tiles(K);
            for (int mt = 0; mt < m2l_tiles(R); ++mt)
                for (int kg = 0; kg < nk; ++kg)
                    for (int lane = 0; lane < 64; ++lane)
                        for (int j = 0; j < 4; ++j) {
                            const int i = 16 * mt + (lane & 15), k = 16 * kg + 4 * j + (lane >> 4);
                            if (i < R && k < K) dst[((size_t)(mt * nk + kg) * 64 + lane) * 4 + j] = a(i, k);
                        }
        };
        // 4x4x1 fragments of an R x K matrix (R, K <= 8), 4-row tiles
        auto put4 = [](double* dst, int R, int K, const std::function<double(int, int)>& a) {
            const int nt4 = (R + 3) / 4, nk4 = (K + 3) / 4;
            for (int t4 = 0; t4 < nt4; ++t4)
                for (int g4 = 0; g4 < nk4; ++g4)
                    for (int lane = 0; lane < 64; ++lane)
                        for (int j = 0; j < 4; ++j) {
                            const int i = 4 * t4 + (lane & 3), k = 4 * g4 + j;
                            if (i < R && k < K) dst[((t4 * nk4 + g4) * 64 + lane) * 4 + j] = a(i, k);
                        }
        };
        std::vector<double> Wu, Wv;
        std::vector<std::vector<double>> Wu3(pb + 1), Wv3(pb + 1);   // stage-3 blocks of one rotation
        for (size_t th = 0; th < thetas.size(); ++th) {
            for (int n = 0; n <= pb; ++n) {
                const double* E = &rot[th * rsz + rot_offset(n)];
                for (int st = 0; st < 2; ++st) {
                    rotation_uv_blocks(E, n, st == 0, Wu, Wv);   // stage 1: E^T, stage 3: E
                    auto wu = [&](int i, int k) { return Wu[(size_t)i * (n + 1) + k]; };
                    // v index m = 1..n; LDS order k' = n - m
                    auto wv = [&](int mi, int mk) { return Wv[(size_t)(mi - 1) * n + (mk - 1)]; };
                    if (st == 0) {
                        double* b = &f1[th * s1];
                        put(b + off1[2 * n], n + 1, n + 1, wu);
                        if (n > 0) put(b + off1[2 * n + 1], n, n, [&](int i, int k) { return wv(n - i, n - k); });
                        if (off1q[2 * n] >= 0) put4(b + off1q[2 * n], n + 1, n + 1, wu);
                        if (off1q[2 * n + 1] >= 0)
                            put4(b + off1q[2 * n + 1], n, n, [&](int i, int k) { return wv(n - i, n - k); });
                    } else {
                        double* b = &f3[th * s3];
                        put(b + off3[2 * n], n + 1, n + 1, wu);
                        if (n > 0)
                            put(b + off3[2 * n + 1], n + 1, n,
                                [&](int i, int k) { return i == 0 ? 0.0 : wv(i, n - k); });
                        Wu3[n] = Wu;
                        Wv3[n] = Wv;
                    }
                }
            }
            double* b3 = &f3[th * s3];
            for (int n1 = 0; n1 <= kM2LPackMax; ++n1)
                for (int n2 = n1 + 1; n1 + n2 <= kM2LPackMax; ++n2) {
                    if (off3p[8 * n1 + n2] < 0) continue;
                    const std::vector<double>&U1 = Wu3[n1], &U2 = Wu3[n2], &V1 = Wv3[n1], &V2 = Wv3[n2];
                    put(b3 + off3p[8 * n1 + n2], 16, n1 + n2 + 2, [&](int i, int k) {
                        if (i < 8) return i <= n1 && k <= n1 ? U1[(size_t)i * (n1 + 1) + k] : 0.0;
                        const int ii = i - 8, kk = k - n1 - 1;
                        return ii <= n2 && kk >= 0 ? U2[(size_t)ii * (n2 + 1) + kk] : 0.0;
                    });
                    // v: row m (0: zero), input k in LDS order (v_m at k = n - m)
                    put(b3 + off3p[8 * n1 + n2] + 256, 16, n1 + n2, [&](int i, int k) {
                        if (i < 8) {
                            if (i == 0 || i > n1 || k >= n1) return 0.0;
                            return V1[(size_t)(i - 1) * n1 + (n1 - k - 1)];
                        }
                        const int ii = i - 8, kk = k - n1;
                        if (ii == 0 || ii > n2 || kk < 0) return 0.0;
                        return V2[(size_t)(ii - 1) * n2 + (n2 - kk - 1)];
                    });
                }
        }
        P.rf_stride1 = s1;
        P.rf_stride3 = s3;
        P.d_rf_off1 = P.upload(off1);
        P.d_rf_off1q = P.upload(off1q);
        P.d_rf_off3 = P.upload(off3);
        P.d_rf_off3p = P.upload(off3p);
        if (P.precision == HFMM_PREC_MIXED) {
            P.d_rf1_32 = P.upload(std::vector<float>(f1.begin(), f1.end()));
            P.d_rf3_32 = P.upload(std::vector<float>(f3.begin(), f3.end()));
        }
        P.d_rf1 = P.upload(f1);   // FP64: M2L, M2M and L2L of FP64 levels
        P.d_rf3 = P.upload(f3);
        if (P.m2l_kernel == 0) {   // the wave kernel's fragments
            const int pc = std::min(pmax, kWave64MaxP);
            P.cr_stride = wave64_rot_regs(pc + 1, 0) * 128;
            std::vector<double> c1((size_t)thetas.size() * P.cr_stride, 0.0), c3(c1.size(), 0.0);
            for (size_t th = 0; th < thetas.size(); ++th)
                for (int n = 0; n <= pc; ++n)
                    for (int st = 0; st < 2; ++st) {
                        rotation_uv_blocks(&rot[th * rsz + rot_offset(n)], n, st == 0, Wu, Wv);
                        double* base = &(st == 0 ? c1 : c3)[th * P.cr_stride];
                        auto at = [&](int h, int i, int k) -> double& {
                            const int j = k / 4;
                            return base[((size_t)(wave64_rot_regs(n, h) + j / 2) * 64 + 16 * (k % 4) + i) * 2 + (j & 1)];
                        };
                        for (int i = 0; i <= n; ++i)
                            for (int k = 0; k <= n; ++k) at(0, i, k) = Wu[(size_t)i * (n + 1) + k];
                        for (int i = 0; i < n; ++i)   // the back table's v rows are the orders 0..n
                            for (int k = 0; k < n; ++k) at(1, st == 0 ? i : i + 1, k) = Wv[(size_t)i * n + k];
                    }
            P.d_cr1 = P.upload(c1);
            P.d_cr3 = P.upload(c3);
            if (P.precision == HFMM_PREC_MIXED) {
                const int pw = std::min(pmax, kWave32MaxP);
                P.wr_stride = kWave32RotFloats;
                std::vector<float> w1((size_t)thetas.size() * P.wr_stride, 0.0f), w3(w1.size(), 0.0f);
                for (size_t th = 0; th < thetas.size(); ++th)
                    for (int n = 1; n <= pw; ++n)
                        for (int st = 0; st < 2; ++st) {
                            rotation_uv_blocks(&rot[th * rsz + rot_offset(n)], n, st == 0, Wu, Wv);
                            float* f = &(st == 0 ? w1 : w3)[th * P.wr_stride];
                            const int qu = n / 4 + 1, qv = (n + 3) / 4;
                            const int u0 = wave32_rot_vecs(0, n), v0 = 64 * kWave32VBlock + wave32_rot_vecs(1, n);
                            for (int k = 0; k <= n; ++k)
                                for (int i = 0; i <= n; ++i)
                                    f[wave32_pos(u0 + qu * k + i / 4, i % 4)] = (float)Wu[(size_t)i * (n + 1) + k];
                            for (int k = 0; k < n; ++k)
                                for (int i = 0; i < n; ++i)
                                    f[wave32_pos(v0 + qv * k + i / 4, i % 4)] = (float)Wv[(size_t)i * n + k];
                            f += kWave32SplitFloats;
                            int v = wave32_joint_vecs(n);
                            for (int k = 0; k <= n; ++k) {
                                for (int i = 0; i <= n; ++i) f[wave32_pos(v + i / 4, i % 4)] = (float)Wu[(size_t)i * (n + 1) + k];
                                v += qu;
                                if (k == 0) continue;
                                for (int i = 0; i < n; ++i) f[wave32_pos(v + i / 4, i % 4)] = (float)Wv[(size_t)i * n + k - 1];
                                v += qv;
                            }
                        }
                P.d_wr1 = P.upload(w1);
                P.d_wr3 = P.upload(w3);
            }
        }
    }
    std::vector<double2> phase((size_t)kNumDirs * (pmax + 1));
    for (int d = 0; d < kNumDirs; ++d)
        for (int m = 0; m <= pmax; ++m)
            phase[(size_t)d * (pmax + 1) + m] = make_double2(std::cos(m * phis[d]), std::sin(m * phis[d]));
    P.d_phase = P.upload(phase);
    if (P.precision == HFMM_PREC_MIXED) {
        std::vector<float2> ph32(phase.size());
        for (size_t i = 0; i < phase.size(); ++i) ph32[i] = make_float2((float)phase[i].x, (float)phase[i].y);
        P.d_phase32 = P.upload(ph32);
    }
    P.d_dinfo = P.upload(dinfo);

    const Gaunt G = make_gaunt(pmax);
    const int D = P.depth;
    // V lists grouped by level / target
    {
        const auto& vt = P.lists.v_tgt;
        const auto& vs = P.lists.v_src;
        for (int L = 2; L <= D; ++L) {
            std::vector<int> targets, ptr{0}, src;
            std::vector<unsigned short> dir;
            for (size_t e = 0; e < vt.size(); ++e) {
                const int tb = vt[e];
                if (t.level[tb] != L) continue;
                if (targets.empty() || targets.back() != tb) {
                    if (!targets.empty()) ptr.push_back((int)src.size());
                    targets.push_back(tb);
                }
                const int sb = vs[e];
                int tx, ty, tz, sx, sy, sz;
                morton_grid(t.code[tb], tx, ty, tz);
                morton_grid(t.code[sb], sx, sy, sz);
                const int dx = tx - sx, dy = ty - sy, dz = tz - sz;
                src.push_back(sb);
                dir.push_back((unsigned short)(kDirV + (dx + 3) * 49 + (dy + 3) * 7 + (dz + 3)));
            }
            if (targets.empty()) continue;
            ptr.push_back((int)src.size());
            XlateLaunch& X = P.m2l[L];
            X.n_targets = (int)targets.size();
            X.targets = P.upload(targets);
            X.ptr = P.upload(ptr);
            X.src = P.upload(src);
            X.dir = P.upload(dir);
            X.ps = X.pt = P.p_level[L];
            X.src_level = X.tgt_level = L;
            X.coax_stride = coax_size(X.pt, X.ps);
            std::vector<double> cx((size_t)dist_d2.size() * X.coax_stride * 2);
            for (size_t i = 0; i < dist_d2.size(); ++i)
                coax_table(0, G, P.k, 2.0 * P.h[L] * std::sqrt((double)dist_d2[i]), P.R[L], P.R[L], X.ps, X.pt,
                           &cx[i * X.coax_stride * 2]);
            X.coax = (double2*)P.upload(cx);
            build_waves(P, P.m2lc[L], 0, L, L, targets, ptr, src, dir, cx, (int)dist_d2.size(), dinfo, P.m2l_fp32[L]);
            if (!P.m2lc[L].use) build_m2l_blocks(P, L, targets, ptr, src, dir, cx, (int)dist_d2.size(), dinfo);
        }
    }
    // M2M (parent level L <- children at L+1) and L2L (parent level L -> children at L+1)
    for (int L = 2; L < D; ++L) {
        std::vector<int> targets, ptr{0}, src;
        std::vector<unsigned short> dir;
        std::vector<int> ctargets, cptr{0}, csrc;
        std::vector<unsigned short> cdir;
        for (int c = t.level_start[L + 1]; c < t.level_start[L + 2]; ++c) {
            const int par = t.parent[c];
            if (targets.empty() || targets.back() != par) {
                if (!targets.empty()) ptr.push_back((int)src.size());
                targets.push_back(par);
            }
            src.push_back(c);
            dir.push_back((unsigned short)(kDirM2M + octant(t.code[c])));
            ctargets.push_back(c);
            csrc.push_back(par);
            cdir.push_back((unsigned short)(kDirL2L + octant(t.code[c])));
            cptr.push_back((int)csrc.size());
        }
        if (targets.empty()) continue;
        ptr.push_back((int)src.size());
        XlateLaunch& A = P.m2m[L];
        A.n_targets = (int)targets.size();
        A.targets = P.upload(targets);
        A.ptr = P.upload(ptr);
        A.src = P.upload(src);
        A.dir = P.upload(dir);
        A.ps = P.p_level[L + 1];
        A.pt = P.p_level[L];
        A.src_level = L + 1;
        A.tgt_level = L;
        A.coax_stride = coax_size(A.pt, A.ps);
        std::vector<double> cx((size_t)A.coax_stride * 2);
        coax_table(1, G, P.k, P.R[L + 1], P.R[L + 1], P.R[L], A.ps, A.pt, cx.data());
        A.coax = (double2*)P.upload(cx);
        const bool up32 = tree_fp32(P, L, 1, targets.size()), down32 = tree_fp32(P, L, 2, targets.size());
        if (!up32) build_waves(P, P.m2mc[L], 1, L + 1, L, targets, ptr, src, dir, cx, 1, dinfo);
        if (!P.m2mc[L].use) build_tree_blocks(P, L, 1, cx, up32);
        XlateLaunch& B = P.l2l[L];
        B.n_targets = (int)ctargets.size();
        B.targets = P.upload(ctargets);
        B.ptr = P.upload(cptr);
        B.src = P.upload(csrc);
        B.dir = P.upload(cdir);
        B.ps = P.p_level[L];
        B.pt = P.p_level[L + 1];
        B.src_level = L;
        B.tgt_level = L + 1;
        B.coax_stride = coax_size(B.pt, B.ps);
        std::vector<double> cy((size_t)B.coax_stride * 2);
        coax_table(2, G, P.k, P.R[L + 1], P.R[L], P.R[L + 1], B.ps, B.pt, cy.data());
        B.coax = (double2*)P.upload(cy);
        if (!down32) build_waves(P, P.l2lc[L], 2, L, L + 1, ctargets, cptr, csrc, cdir, cy, 1, dinfo);
        if (!P.l2lc[L].use) build_tree_blocks(P, L, 2, cy, down32);
    }
}

P2PArgs p2p_args(const hfmm_plan& P, int out_mode, double2* out);

// Near-field work items.  A leaf's targets go in chunks of up to 64 R (R per lane of a wave); a
// remainder that is not a power of two (and above 4 R) goes as its largest power of two first, so
// that few target slots of the R x L lanes are idle.  Chunks of more than `limit` pairs are halved,
// down to 16 targets (each chunk stages the leaf's sources once more: about a tenth of the work of
// 16 targets).
struct NearWork {
    std::vector<NearItem> items;
    std::vector<int> prob;
    std::vector<int64_t> cost;
    void add(const Tree& t, const std::vector<int>& leaf_box, const std::vector<int>& total, int l0, int l1, int R,
             int64_t limit, int problem) {
        for (int l = l0; l < l1; ++l) {
            const int b = leaf_box[l], n = t.count[b];
            int cap = 16;
            while (2 * cap <= 64 * R && (int64_t)2 * cap * total[l] <= limit) cap *= 2;
            for (int t0 = 0, c = 0; t0 < n; t0 += c) {
                c = std::min(n - t0, 64 * R);
                if (c < 64 * R && c > 4 * R)
                    while (c & (c - 1)) c &= c - 1;   // the largest power of two
                c = std::min(c, cap);
                items.push_back({l, b, t.pstart[b] + t0, c});
                prob.push_back(problem);
                cost.push_back((int64_t)(c + 8) * total[l] + 4096);
            }
        }
    }
    // Interleaved for the XCDs (workgroup i runs on XCD i % kXcds): XCD x takes a contiguous
    // range of the (Morton ordered) items, so that its L2 holds one region's points, with 1 / 8 of
    // the cost; within it the longest first, by powers of two.  Padded with empty items.
    std::pair<std::vector<NearItem>, std::vector<int>> ordered() const {
        int64_t sum = 0, acc = 0;
        for (int64_t c : cost) sum += c;
        std::vector<int> of[kXcds];
        for (size_t i = 0; i < items.size(); ++i) {
            of[std::min<int64_t>(kXcds - 1, (acc + cost[i] / 2) * kXcds / std::max<int64_t>(1, sum))].push_back((int)i);
            acc += cost[i];
        }
        size_t most = 0;
        for (auto& v : of) {
            std::stable_sort(v.begin(), v.end(), [&](int x, int y) { return ilogb_cost(x) > ilogb_cost(y); });
            most = std::max(most, v.size());
        }
        std::pair<std::vector<NearItem>, std::vector<int>> out;
        out.first.assign(most * kXcds, NearItem{0, 0, 0, 0});
        out.second.assign(most * kXcds, 0);
        for (int x = 0; x < kXcds; ++x)
            for (size_t i = 0; i < of[x].size(); ++i) {
                out.first[i * kXcds + x] = items[of[x][i]];
                out.second[i * kXcds + x] = prob[of[x][i]];
            }
        return out;
    }
    int ilogb_cost(int i) const { return 63 - __builtin_clzll((unsigned long long)cost[i]); }
};

// Pairs up to which a chunk stays whole: a thousandth of those of the launch, a quarter of a
// SIMD's share on each of the kNearWaves that take it.
int64_t near_pairs(const std::vector<int>& leaf_box, const std::vector<int>& total, const Tree& t, int l0, int l1) {
    int64_t pairs = 0;
    for (int l = l0; l < l1; ++l) pairs += (int64_t)total[l] * t.count[leaf_box[l]];
    return pairs;
}
int64_t near_limit(int64_t pairs) { return pairs / 1024; }

void build_p2p(hfmm_plan& P) {
    const Tree& t = P.tree;
    const Lists& ls = P.lists;
    const int nb = t.n_boxes();
    auto csr = [nb](const std::vector<int>& tg, const std::vector<int>& sr, std::vector<int>& ptr, std::vector<int>& s) {
        ptr.assign(nb + 1, 0);
        for (int x : tg) ptr[x + 1]++;
        for (int i = 0; i < nb; ++i) ptr[i + 1] += ptr[i];
        s.assign(sr.size(), 0);
        std::vector<int> pos(ptr.begin(), ptr.end() - 1);
        for (size_t e = 0; e < tg.size(); ++e) s[pos[tg[e]]++] = sr[e];
    };
    std::vector<int> up, us, wp, ws, xp, xs;
    csr(ls.u_tgt, ls.u_src, up, us);
    csr(ls.w_tgt, ls.w_src, wp, ws);
    csr(ls.x_tgt, ls.x_src, xp, xs);
    // box centre and half diagonal, for the bound on k r over a leaf's pairs
    auto geom = [&](int b, double c[3]) {
        int g[3];
        morton_grid(t.code[b], g[0], g[1], g[2]);
        const double w = t.extent * std::ldexp(1.0, -t.level[b]);
        for (int a = 0; a < 3; ++a) c[a] = (g[a] + 0.5) * w + t.pmin[a];
        return 0.5 * std::sqrt(3.0) * w;
    };
    // leaves whose pairs stay within k r <= kP2PFp32MaxKr first (FP32 near field), then the
    // rest (FP32 with the phase in FP64); Morton order within each class
    std::vector<int> leaves[2];
    double kr_max = 0.0;
    for (int b = 0; b < nb; ++b) {
        if (!t.is_leaf[b]) continue;
        double kr = 0.0;
        if (P.precision == HFMM_PREC_MIXED) {
            double cb[3], cs[3];
            const double hb = geom(b, cb);
            auto reach = [&](int box) {
                const double hs = geom(box, cs);
                const double d = std::sqrt((cb[0] - cs[0]) * (cb[0] - cs[0]) + (cb[1] - cs[1]) * (cb[1] - cs[1]) +
                                           (cb[2] - cs[2]) * (cb[2] - cs[2]));
                kr = std::max(kr, P.k * (d + hb + hs));
            };
            reach(b);
            for (int e = up[b]; e < up[b + 1]; ++e) reach(us[e]);
            for (int e = wp[b]; e < wp[b + 1]; ++e) reach(ws[e]);
            for (int a = b; a >= 0; a = t.parent[a])
                for (int e = xp[a]; e < xp[a + 1]; ++e) reach(xs[e]);
        }
        leaves[kr > kP2PFp32MaxKr].push_back(b);
        kr_max = std::max(kr_max, kr);
    }
    P.n_p2p_fp32 = (int)leaves[0].size();
    P.p2p_lowk = P.precision == HFMM_PREC_MIXED && kr_max <= kP2PLowKr;
    std::vector<int> leaf_box, batch_ptr{0}, rng_delta, total;
    std::vector<NearBatch> batches;
    std::vector<double> floor2;
    std::vector<int> far_leaves;
    int64_t pairs = 0;
    for (int b = 0; b < nb; ++b)
        if (t.is_leaf[b] && t.level[b] >= 2) far_leaves.push_back(b);
    for (int cls = 0; cls < 2; ++cls)
        for (int b : leaves[cls]) {
            leaf_box.push_back(b);
            int acc = 0;
            double src_maxabs = 0.0;
            const size_t batch0 = batches.size();
            // a range of the leaf's sources: its start in the batch it begins in, and the batches
            // that begin within it
            auto add = [&](int box) {
                src_maxabs = std::max(src_maxabs, P.box_maxabs[box]);
                if (t.count[box] == 0) return;
                const int range = (int)rng_delta.size();
                rng_delta.push_back(t.pstart[box] - acc);
                if (acc % 64) batches[batch0 + acc / 64].mask |= 1ull << (acc % 64);
                acc += t.count[box];
                while ((int)(batches.size() - batch0) * 64 < acc) batches.push_back({0, range, 0});
            };
            add(b);
            for (int e = up[b]; e < up[b + 1]; ++e) add(us[e]);
            for (int e = wp[b]; e < wp[b + 1]; ++e) add(ws[e]);
            for (int a = b; a >= 0; a = t.parent[a])
                for (int e = xp[a]; e < xp[a + 1]; ++e) add(xs[e]);
            batch_ptr.push_back((int)batches.size());
            total.push_back(acc);
            // the reference's coincidence floor (jaxfmm/near.py:252-261, "pair" form in FP64):
            // pairs with r <= 16 eps (max |x_t| + max |x_s|) contribute nothing
            const double fl = 16.0 * std::numeric_limits<double>::epsilon() * (P.box_maxabs[b] + src_maxabs);
            floor2.push_back(fl * fl);
            pairs += (int64_t)acc * t.count[b];
        }
    P.n_leaves = (int)leaf_box.size();
    P.n_far_leaves = (int)far_leaves.size();
    P.n_p2p_pairs = pairs;
    P.d_leaf_box = P.upload(leaf_box);
    P.d_far_leaves = P.upload(far_leaves);
    P.d_batch_ptr = P.upload(batch_ptr);
    P.d_batches = P.upload(batches);
    P.d_rng_delta = P.upload(rng_delta);
    P.d_leaf_src_total = P.upload(total);
    P.d_floor2 = P.upload(floor2);
    P.box_maxabs = std::vector<double>();
    for (int cls = 0; cls < 2; ++cls) {
        const int l0 = cls ? P.n_p2p_fp32 : 0, l1 = cls ? P.n_leaves : P.n_p2p_fp32;
        const int R = P.precision == HFMM_PREC_FP64 ? kP2PFp64TargetsPerLane : P.p2p_tile;
        for (auto& [dst, r] : {std::make_pair(&P.near_items[cls], R),
                               std::make_pair(&P.field_items[cls], kP2PFieldTargetsPerLane)}) {
            NearWork w;
            w.add(t, leaf_box, total, l0, l1, r, near_limit(near_pairs(leaf_box, total, t, l0, l1)), 0);
            const std::vector<NearItem> items = w.ordered().first;
            dst->n = (int)items.size();
            dst->items = P.upload(items);
        }
    }
    if (P.in_batch) {
        P.leaf_box = std::move(leaf_box);
        P.leaf_total = std::move(total);
    }
    // FP32-phase leaves whose estimated error from FP32 coordinate differences is within
    // p2p_coord32_tol take them (the check runs once, on the GPU, in FP64)
    if (P.precision == HFMM_PREC_MIXED && !P.p2p_lowk && P.p2p_coord32_tol > 0.0 && P.n_p2p_fp32 > 0) {
        P.d_coord32 = P.alloc<unsigned char>(P.n_leaves);
        HIPCHK(hipMemset(P.d_coord32, 0, P.n_leaves));
        launch_p2p_coord_check(p2p_args(P, 0, nullptr), P.n_p2p_fp32, P.p2p_coord32_tol, P.d_coord32, P.stream);
        std::vector<unsigned char> f(P.n_leaves);
        HIPCHK(hipMemcpyAsync(f.data(), P.d_coord32, P.n_leaves, hipMemcpyDeviceToHost, P.stream));
        HIPCHK(hipStreamSynchronize(P.stream));
        for (unsigned char v : f) P.n_leaves_coord32 += v;
    }
}

size_t wave_part_bytes(const M2LWaveLevel& B, int n_slots) {
    const int p = std::max(B.ps, B.pt);
    return (size_t)n_slots * B.tb *
           (B.fp32 ? 2 * (p + 1) * (p + 1) * sizeof(float) : 4 * wave64_regs(p) * sizeof(double4));
}

// The partial sums of the wave kernels' split blocks: one buffer for all levels, which run one after
// another (FP64, 16 targets a block: up to 132 MB at p = 10, 226 MB at p = 14).  Allocated with the plan;
// a plan of a batch, which has a buffer for all its problems, gets its own when it is first evaluated
// alone (64 problems of 2k to 200k points in FP64: 9.3 GB with a buffer each, 2.7 GB without).
void alloc_wave_parts(hfmm_plan& P) {
    size_t most = 0;
    for (const M2LWaveLevel& B : P.m2lc)
        if (!B.part) most = std::max(most, wave_part_bytes(B, B.n_slots));
    if (!most) return;
    void* all = P.alloc<char>(most);
    for (M2LWaveLevel& B : P.m2lc)
        if (B.n_slots) B.part = all;
}

void build_plan(hfmm_plan& P, const double* xyz, int64_t n, double k, const hfmm_opts& o) {
    if (!std::isfinite(k)) fail(HFMM_ERR_ARG, "k must be a finite real number");
    if (n <= 0 || n > (int64_t)1 << 30) fail(HFMM_ERR_ARG, "positions must be a nonempty finite (N,3) array");
    for (int64_t i = 0; i < 3 * n; ++i)
        if (!std::isfinite(xyz[i])) fail(HFMM_ERR_ARG, "positions must be a nonempty finite (N,3) array");
    if (o.p < 2 || o.n_max < 1) fail(HFMM_ERR_ARG, "p must be an integer >=2; N_max must be a positive integer");
    if (o.p > kMaxP) fail(HFMM_ERR_ARG, "p exceeds the supported maximum of 40");
    for (int L = 0; L < HFMM_MAX_LEVELS; ++L)
        if (o.p_level[L] != 0 && (o.p_level[L] < 2 || o.p_level[L] > kMaxP))
            fail(HFMM_ERR_ARG, "p_level entries must be 0 or in [2, 40]");
    if (o.precision != HFMM_PREC_FP64 && o.precision != HFMM_PREC_MIXED) fail(HFMM_ERR_ARG, "unknown precision");
    if (o.m2l_kernel != 0 && o.m2l_kernel != 1 && o.m2l_kernel != 8 && o.m2l_kernel != 16 && o.m2l_kernel != 32 &&
        o.m2l_kernel != 64)
        fail(HFMM_ERR_ARG, "m2l_kernel must be 0, 1, 8, 16, 32 or 64");
    if (o.p2p_tile != 0 && o.p2p_tile != 1 && o.p2p_tile != 2 && o.p2p_tile != 4)
        fail(HFMM_ERR_ARG, "p2p_tile must be 0, 1, 2 or 4");
    check_device();
    upload_legendre_coefficients();
    P.n = n;
    P.k = std::fabs(k);
    P.conj = k < 0;
    P.precision = o.precision;
    P.use_graph = o.use_graph;
    P.m2l_kernel = o.m2l_kernel;
    P.p2p_tile = o.p2p_tile == 0 ? 2 : o.p2p_tile;
    if (!std::isfinite(o.p2p_coord32_tol)) fail(HFMM_ERR_ARG, "p2p_coord32_tol must be a finite number");
    P.p2p_coord32_tol = o.p2p_coord32_tol == 0.0 ? HFMM_P2P_COORD32_TOL : o.p2p_coord32_tol;
    {
        int dev = 0, lds = 65536;
        HIPCHK(hipGetDevice(&dev));
        if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && lds > 0)
            P.max_lds = (size_t)lds;
    }
    if (o.tree_device) {
        build_tree_device(xyz, n, o.n_max, o.max_depth, P.tree, P.lists);
    } else {
        P.tree = build_tree(xyz, n, o.n_max, o.max_depth);
        P.lists = build_lists(P.tree);
    }
    const Tree& t = P.tree;
    P.depth = t.depth;
    P.pmax = 0;
    for (int L = 0; L < kMaxLevels; ++L) {
        P.p_level[L] = (L < HFMM_MAX_LEVELS && o.p_level[L] > 0) ? o.p_level[L] : o.p;
        P.h[L] = t.extent * std::ldexp(1.0, -(L + 1));
        P.R[L] = std::sqrt(3.0) * P.h[L];
        if (L >= 1 && L <= t.depth) P.pmax = std::max(P.pmax, P.p_level[L]);
        P.p_eff[L] = P.p_level[L];
        const double kd = P.k * 2.0 * P.R[L];   // k times the box diagonal
        P.m2l_fp32[L] = o.precision == HFMM_PREC_MIXED &&
                        (o.m2l_fp64_levels < 0 ? kd <= HFMM_MIXED_FP32_MAX_KD : !((o.m2l_fp64_levels >> L) & 1));
    }
    HIPCHK(hipStreamCreateWithFlags(&P.stream, hipStreamNonBlocking));
    // sorted positions (SoA, FP64) and permutation
    std::vector<double> X(n), Y(n), Z(n);
    std::vector<int> perm(n);
    for (int64_t i = 0; i < n; ++i) {
        const int64_t o2 = t.perm[i];
        X[i] = xyz[3 * o2];
        Y[i] = xyz[3 * o2 + 1];
        Z[i] = xyz[3 * o2 + 2];
        perm[i] = (int)o2;
    }
    P.dX = P.upload(X);
    P.dY = P.upload(Y);
    P.dZ = P.upload(Z);
    P.d_perm = P.upload(perm);
    // boxes
    const int nb = t.n_boxes();
    // largest |x| per box (points of leaves, then children into parents: boxes are in level
    // order, so children come after their parents), for the near field's coincidence floor
    P.box_maxabs.assign(nb, 0.0);
    for (int b = nb - 1; b >= 0; --b) {
        if (t.is_leaf[b])
            for (int i = t.pstart[b]; i < t.pstart[b] + t.count[b]; ++i)
                P.box_maxabs[b] = std::max(P.box_maxabs[b], std::sqrt(X[i] * X[i] + Y[i] * Y[i] + Z[i] * Z[i]));
        if (t.parent[b] >= 0) P.box_maxabs[t.parent[b]] = std::max(P.box_maxabs[t.parent[b]], P.box_maxabs[b]);
    }
    std::vector<double> centre(3 * (size_t)nb);
    P.exp_off.assign(nb, 0);
    P.sd_off.assign(nb, 0);
    P.sd32_off.assign(nb, 0);
    int64_t off = 0;
    for (int b = 0; b < nb; ++b) {
        int gx, gy, gz;
        morton_grid(t.code[b], gx, gy, gz);
        const double s = t.extent * std::ldexp(1.0, -t.level[b]);
        const double half = t.extent * std::ldexp(1.0, -(t.level[b] + 1));
        centre[3 * b] = gx * s + half + t.pmin[0];
        centre[3 * b + 1] = gy * s + half + t.pmin[1];
        centre[3 * b + 2] = gz * s + half + t.pmin[2];
        P.exp_off[b] = off;
        off += ncoef(P.p_level[t.level[b]]);
        if (b == 0) P.n_sd = wave_sd_pad(P.pmax);
        P.sd_off[b] = P.n_sd;
        const int entries = (P.p_level[t.level[b]] + 1) * (P.p_level[t.level[b]] + 2) / 2;
        P.n_sd += entries;
        if (b == 0) P.n_sd32 = wave32_sd_pad(P.pmax);
        P.sd32_off[b] = P.n_sd32;
        P.n_sd32 += (entries + 1) / 2;
    }
    P.n_coef = off;
    P.d_centre = P.upload(centre);
    P.d_level = P.upload(t.level);
    P.d_pstart = P.upload(t.pstart);
    P.d_count = P.upload(t.count);
    P.d_expoff = P.upload(P.exp_off);
    std::vector<int> pl(P.p_level, P.p_level + kMaxLevels);
    std::vector<double> rl(P.R, P.R + kMaxLevels);
    P.d_plevel = P.upload(pl);
    P.d_R = P.upload(rl);
    build_p2p(P);
    {
        // P2M / L2P descriptors of the far leaves, in the order of d_far_leaves
        std::vector<LeafDesc> ld;
        for (int b = 0; b < nb; ++b)
            if (t.is_leaf[b] && t.level[b] >= 2) {
                LeafDesc d{};
                d.box = b;
                d.level = t.level[b];
                d.pstart = t.pstart[b];
                d.count = t.count[b];
                d.exp_off = P.exp_off[b];
                d.cx = centre[3 * b];
                d.cy = centre[3 * b + 1];
                d.cz = centre[3 * b + 2];
                ld.push_back(d);
            }
        if ((int)ld.size() != P.n_far_leaves) fail(HFMM_ERR_INTERNAL, "far leaf descriptors out of step");
        P.d_leafdesc = P.upload(ld);
    }
    build_tables(P);
    // P2M: points staged per pass, sized for the largest leaf degree
    P.p_leafmax = 2;
    for (int b = 0; b < t.n_boxes(); ++b)
        if (t.is_leaf[b]) P.p_leafmax = std::max(P.p_leafmax, P.p_level[t.level[b]]);
    P.p2m_chunk = p2m_chunk(P.p_leafmax);
    for (int l = 2, first = 0; l <= P.depth; ++l) {   // the far leaves are ordered by level
        int n = 0;
        for (int b = t.level_start[l]; b < t.level_start[l + 1]; ++b) n += t.is_leaf[b] ? 1 : 0;
        if (!n) continue;
        if (!P.l2p_runs.empty() && (P.l2p_runs.back().p == P.p_level[l] || P.l2p_runs.back().n < kL2PRunLeaves ||
                                    P.n_far_leaves - first < kL2PRunLeaves)) {
            P.l2p_runs.back().n += n;
            P.l2p_runs.back().p = std::max(P.l2p_runs.back().p, P.p_level[l]);
        } else {
            P.l2p_runs.push_back({first, n, P.p_level[l]});
        }
        first += n;
    }
    P.dM = P.alloc<double2>(P.n_coef);
    bool any_fp32 = false, any_l2l32 = false;
    for (int L = 0; L < kMaxLevels; ++L) {
        any_fp32 = any_fp32 || (P.m2lb[L].use && P.m2lb[L].fp32) || (P.m2mb[L].use && P.m2mb[L].fp32);
        any_l2l32 = any_l2l32 || (P.l2lb[L].use && P.l2lb[L].fp32);
    }
    if (any_fp32) P.dM32 = P.alloc<float2>(P.n_coef);
    P.dL = P.alloc<double2>(P.n_coef);
    if (any_l2l32) P.dL32 = P.alloc<float2>(P.n_coef);
    bool any_col = false, any_l2l_col = false, any_wave32 = false;
    for (int L = 0; L < kMaxLevels; ++L) {
        any_col = any_col || (P.m2lc[L].use && !P.m2lc[L].fp32) || P.m2mc[L].use;
        any_wave32 = any_wave32 || (P.m2lc[L].use && P.m2lc[L].fp32);
        any_l2l_col = any_l2l_col || P.l2lc[L].use;
    }
    if (!P.in_batch) alloc_wave_parts(P);
    const size_t n_sd = P.n_sd + wave_sd_pad(P.pmax);
    for (double4** buf : {any_col ? &P.dMs : nullptr, any_l2l_col ? &P.dLs : nullptr})
        if (buf) {
            *buf = P.alloc<double4>(n_sd);
            HIPCHK(hipMemset(*buf, 0, n_sd * sizeof(double4)));
        }
    if (any_wave32) {
        const size_t n32 = 2 * (P.n_sd32 + wave32_sd_pad(P.pmax));
        P.dMs32 = P.alloc<float4>(n32);
        HIPCHK(hipMemset(P.dMs32, 0, n32 * sizeof(float4)));
    }
    P.d_q = P.alloc<double2>(n);
    P.d_far = P.alloc<double2>(n);
    P.d_qin = P.alloc<double2>(n);
    P.d_out = P.alloc<double2>(n);
    HIPCHK(hipDeviceSynchronize());
}

XlateArgs xargs(const hfmm_plan& P, const XlateLaunch& X, const double2* srcbuf, double2* dstbuf, int accumulate) {
    XlateArgs a;
    a.targets = X.targets;
    a.ptr = X.ptr;
    a.src = X.src;
    a.dir = X.dir;
    a.dinfo = P.d_dinfo;
    a.phase = P.d_phase;
    a.rot = P.d_rot;
    a.coax = X.coax;
    a.coax_stride = X.coax_stride;
    a.ps = P.p_eff[X.src_level];
    a.pt = P.p_eff[X.tgt_level];
    a.tps = X.ps;
    a.tpt = X.pt;
    a.pmax = P.pmax;
    a.accumulate = accumulate;
    a.split = 1;
    a.srcbuf = srcbuf;
    a.dstbuf = dstbuf;
    a.exp_off = P.d_expoff;
    return a;
}

M2LBlockArgs block_args(const hfmm_plan& P, const M2LBlockLevel& B, bool fp32, const void* src, double2* dst,
                        int overwrite) {
    M2LBlockArgs a;
    a.p = P.p_eff[B.src_level];
    a.p_tab = B.ps;
    a.pt = P.p_eff[B.tgt_level];
    a.pt_tab = B.pt;
    a.overwrite = overwrite;
    a.n_items = B.n_items;
    a.items = B.items;
    a.blk_targets = B.targets;
    a.grp_dir = B.dir;
    a.grp_off = B.off;
    a.units1 = B.units1;
    a.n_units1 = B.n_units1;
    a.units2 = B.units2;
    a.n_units2 = B.n_units2;
    a.units3 = B.units3;
    a.n_units3 = B.n_units3;
    a.rot1 = fp32 ? (const void*)P.d_rf1_32 : (const void*)P.d_rf1;
    a.rot3 = fp32 ? (const void*)P.d_rf3_32 : (const void*)P.d_rf3;
    a.rot_off1 = P.d_rf_off1;
    a.rot_off1q = P.d_rf_off1q;
    a.rot_off3 = P.d_rf_off3;
    a.rot_off3p = P.d_rf_off3p;
    a.rot_stride1 = P.rf_stride1;
    a.rot_stride3 = P.rf_stride3;
    a.phase = fp32 ? (const void*)P.d_phase32 : (const void*)P.d_phase;
    a.phase_stride = P.pmax + 1;
    a.dinfo = P.d_dinfo;
    a.coax = B.coax;
    a.coax_off = B.coax_off;
    a.coax_offq = B.coax_offq;
    a.coax_stride = B.coax_stride;
    a.M = src;
    a.L = dst;
    a.exp_off = P.d_expoff;
    return a;
}

M2LWaveArgs wave_args(const hfmm_plan& P, const M2LWaveLevel& B, const void* src, double2* dst, int overwrite) {
    M2LWaveArgs a;
    a.ps = P.p_eff[B.src_level];
    a.pt = P.p_eff[B.tgt_level];
    a.overwrite = overwrite;
    a.n_items = B.n_items;
    a.items = B.items;
    a.n_blocks = B.n_blocks;
    a.part = B.n_slots ? B.part : nullptr;
    a.part_ptr = B.part_ptr;
    a.tb = B.tb;
    a.blk_targets = B.targets;
    a.grp_class = B.cls;
    a.grp_src = B.src;
    a.grp_dir = B.dir;
    const int layout = wave32_wpe(std::max(a.ps, a.pt)) == 1 ? kWave32SplitFloats : 0;
    a.rot1 = B.fp32 ? (const void*)(P.d_wr1 + layout) : P.d_cr1;
    a.rot3 = B.fp32 ? (const void*)(P.d_wr3 + layout) : P.d_cr3;
    a.rot_stride = B.fp32 ? P.wr_stride : P.cr_stride;
    a.phase = B.fp32 ? (const void*)P.d_phase32 : P.d_phase;
    a.phase_stride = P.pmax + 1;
    a.coax = B.coax;
    a.coax_stride = B.coax_stride;
    a.M = src;
    a.L = dst;
    a.exp_off = P.d_expoff;
    return a;
}

const void* wave_source(const hfmm_plan& P, const M2LWaveLevel& B) {
    return B.fp32 ? (const void*)P.dMs32 : P.dMs;
}

void launch_wave(const hfmm_plan& P, const M2LWaveLevel& B, const void* src, double2* dst, int overwrite,
                 hipStream_t s) {
    const M2LWaveArgs a = wave_args(P, B, src, dst, overwrite);
    (B.fp32 ? launch_m2l_wave32 : launch_m2l_wave64)(a, std::max(a.ps, a.pt), s);
}

// parts of one evaluate's device sequence (a batch runs them for all problems, with the
// matrix-core M2L and the near field as launches over the work of every problem)
constexpr int kSeqUp = 1;          // charges, clears, P2M, M2M
constexpr int kSeqM2LGeneric = 2;  // M2L levels on the generic kernel
constexpr int kSeqM2LBlock = 4;    // M2L levels on the matrix-core block kernel
constexpr int kSeqDown = 8;        // L2L, L2P
constexpr int kSeqP2P = 16;        // near field and output
constexpr int kSeqAll = 31;

// first coefficient of the expansions of tree level l (boxes are in level order); n_coef
// past the deepest level
int64_t level_coef(const hfmm_plan& P, int l) {
    const Tree& t = P.tree;
    if (l > t.depth) return P.n_coef;
    const int b = t.level_start[l];
    return b < t.n_boxes() ? P.exp_off[b] : P.n_coef;
}

// the expansions of level l in (S, D) form, x basis buffer e to sd
void level_to_sd(const hfmm_plan& P, int l, const double2* e, double4* sd, hipStream_t s) {
    const Tree& t = P.tree;
    const int b0 = t.level_start[l], b1 = t.level_start[l + 1];
    if (b1 > b0) launch_to_sd64(e + P.exp_off[b0], sd + P.sd_off[b0], b1 - b0, P.p_level[l], s);
}

// Runs of levels of one precision and table degree whose M2L the wave kernels take, less the FP64
// levels that M2M has in (S, D) form already.  A run is contiguous in both buffers: one launch.  (A launch per
// level made the upward passes of 64 problems of 30 points, which are launches alone, 10% longer.)
struct LevelRun {
    int b0, n, p;
    bool fp32;
};
std::vector<LevelRun> sd_runs(const hfmm_plan& P) {
    const Tree& t = P.tree;
    auto needed = [&](int l, bool fp32) {
        return l <= P.depth && P.m2lc[l].use && P.m2lc[l].fp32 == fp32 && (fp32 || !P.m2mc[l - 1].use);
    };
    std::vector<LevelRun> runs;
    for (int l = 2; l <= P.depth;) {
        const bool fp32 = P.m2lc[l].fp32;
        if (!needed(l, fp32)) {
            ++l;
            continue;
        }
        const int b0 = t.level_start[l], p = P.p_level[l];
        while (needed(l, fp32) && P.p_level[l] == p) ++l;
        runs.push_back({b0, t.level_start[l] - b0, p, fp32});
    }
    return runs;
}

int out_mode_of(const hfmm_plan& P, int q_type) {
    return (P.conj ? 1 : 0) | ((P.k == 0.0 && real_charges(q_type)) ? 2 : 0);
}

P2PArgs p2p_args(const hfmm_plan& P, int out_mode, double2* out) {
    P2PArgs pa{};
    pa.leaf_box = P.d_leaf_box;
    pa.bx = P.boxes();
    pa.batch_ptr = P.d_batch_ptr;
    pa.batches = P.d_batches;
    pa.rng_delta = P.d_rng_delta;
    pa.leaf_src_total = P.d_leaf_src_total;
    pa.floor2 = P.d_floor2;
    pa.X = P.dX;
    pa.Y = P.dY;
    pa.Z = P.dZ;
    pa.q = P.d_q;
    pa.k = P.k;
    const nearfield::HalfTurnK kp = nearfield::halfturn_k(P.k);
    pa.kp_hi = kp.hi;
    pa.kp_lo = kp.lo;
    pa.far = P.d_far;
    pa.perm = P.d_perm;
    pa.out_mode = out_mode;
    pa.out = out;
    pa.coord32 = P.d_coord32;
    return pa;
}

// The device sequence of one evaluate (the parts selected).  ev (optional, 8 entries)
// brackets the phases; lev (optional, 2 per level) brackets the M2L launch of every level.
// field (optional): E = -grad phi, 3 complex values per point in input order.
void run_sequence(hfmm_plan& P, const void* q, int q_type, double2* out, hipStream_t s, hipEvent_t* ev,
                  hipEvent_t* lev = nullptr, double2* field = nullptr, int parts = kSeqAll) {
    auto mark = [&](int i) {
        if (ev) HIPCHK(hipEventRecord(ev[i], s));
    };
    const DevBoxes bx = P.boxes();
    const DevLevels lv = P.levels();
    if (parts & kSeqUp) {
        mark(0);
        launch_gather_charges(q, q_type, P.d_perm, P.n, P.conj, P.d_q, s);
        launch_fill_zero(P.dL, P.n_coef, s);
        launch_fill_zero(P.d_far, P.n, s);
        mark(1);
        launch_p2m(P.d_leafdesc, P.n_far_leaves, P.p2m_chunk, lv, P.dX, P.dY, P.dZ, P.d_q, P.k, P.p_leafmax, P.dM, s);
        mark(2);
        bool conv[kMaxLevels + 1] = {};   // levels whose multipoles are in FP32 already
        for (int L = P.depth - 1; L >= 2; --L) {
            if (P.m2mc[L].use) {
                const M2LWaveLevel& B = P.m2mc[L];
                level_to_sd(P, L + 1, P.dM, P.dMs, s);
                launch_wave(P, B, P.dMs, P.dM, 1, s);
            } else if (P.m2mb[L].use) {
                const M2LBlockLevel& B = P.m2mb[L];
                if (B.fp32) {   // the children's multipoles (complete now) in FP32
                    const int64_t c0 = level_coef(P, L + 1), c1 = level_coef(P, L + 2);
                    launch_to_float(P.dM + c0, P.dM32 + c0, c1 - c0, s);
                    conv[L + 1] = true;
                }
                if (B.split) launch_zero_boxes(B.zero, B.n_zero, P.d_expoff, ncoef(P.p_eff[L]), P.dM, s);
                launch_m2l_block(block_args(P, B, B.fp32, B.fp32 ? (const void*)P.dM32 : (const void*)P.dM, P.dM,
                                            B.split ? 0 : 1),
                                 B.tb, B.grp, B.fp32, s);
            }
            else if (P.m2m[L].n_targets)
                launch_xlate(xargs(P, P.m2m[L], P.dM, P.dM, 0), P.m2m[L].n_targets, s);
        }
        mark(3);
        if (parts & kSeqM2LBlock)   // (a batch converts those of all its plans at once)
            for (const LevelRun& r : sd_runs(P)) {
                if (r.fp32)
                    launch_to_sd32(P.dM + P.exp_off[r.b0], P.dMs32 + 2 * P.sd32_off[r.b0], r.n, r.p, s);
                else
                    launch_to_sd64(P.dM + P.exp_off[r.b0], P.dMs + P.sd_off[r.b0], r.n, r.p, s);
            }
        // multipoles in FP32 for the FP32 block levels: every level not converted for an FP32
        // M2M (the converted ones need not be contiguous), one launch per run of levels
        bool any_fp32 = false;
        for (int L = 2; L <= P.depth; ++L) any_fp32 |= P.m2l[L].n_targets && P.m2lb[L].use && P.m2lb[L].fp32;
        if (any_fp32)
            for (int l0 = 0; l0 <= P.depth;) {
                if (conv[l0]) {
                    ++l0;
                    continue;
                }
                int l1 = l0;
                while (l1 + 1 <= P.depth && !conv[l1 + 1]) ++l1;
                const int64_t c0 = level_coef(P, l0), c1 = level_coef(P, l1 + 1);
                launch_to_float(P.dM + c0, P.dM32 + c0, c1 - c0, s);
                l0 = l1 + 1;
            }
    }
    for (int L = 2; L <= P.depth; ++L) {
        if (!P.m2l[L].n_targets) continue;
        const M2LBlockLevel& B = P.m2lb[L];
        if (P.m2lc[L].use) {
            if (!(parts & kSeqM2LBlock)) continue;
            if (lev) HIPCHK(hipEventRecord(lev[2 * L], s));
            launch_wave(P, P.m2lc[L], wave_source(P, P.m2lc[L]), P.dL, P.m2lc[L].fp32, s);
            if (lev) HIPCHK(hipEventRecord(lev[2 * L + 1], s));
            continue;
        }
        if (!B.use) {
            if (!(parts & kSeqM2LGeneric)) continue;
            if (lev) HIPCHK(hipEventRecord(lev[2 * L], s));
            // coarse levels with few targets (degrees above the matrix-core kernel's): the
            // source lists split over up to 16 workgroups per target, so that about 2048
            // workgroups fill the GPU (level 2 of a uniform tree has 64 targets)
            XlateArgs a = xargs(P, P.m2l[L], P.dM, P.dL, 1);
            a.split = std::max(1, std::min(16, 2048 / std::max(1, P.m2l[L].n_targets)));
            launch_xlate(a, P.m2l[L].n_targets, s);
            if (lev) HIPCHK(hipEventRecord(lev[2 * L + 1], s));
            continue;
        }
        if (!(parts & kSeqM2LBlock)) continue;
        const M2LBlockArgs a =
            block_args(P, B, B.fp32, B.fp32 ? (const void*)P.dM32 : (const void*)P.dM, P.dL, 0);
        if (lev) HIPCHK(hipEventRecord(lev[2 * L], s));
        launch_m2l_block(a, B.tb, B.grp, B.fp32, s);
        if (lev) HIPCHK(hipEventRecord(lev[2 * L + 1], s));
    }
    if (parts & (kSeqM2LGeneric | kSeqM2LBlock)) mark(4);
    const int out_mode = out_mode_of(P, q_type);
    if (parts & kSeqDown) {
        for (int L = 2; L < P.depth; ++L) {
            const M2LBlockLevel& B = P.l2lb[L];
            if (P.l2lc[L].use) {
                level_to_sd(P, L, P.dL, P.dLs, s);
                launch_wave(P, P.l2lc[L], P.dLs, P.dL, 0, s);
            } else if (B.use && B.fp32) {   // the parents' locals (complete now) in FP32
                const int64_t c0 = level_coef(P, L), c1 = level_coef(P, L + 1);
                launch_to_float(P.dL + c0, P.dL32 + c0, c1 - c0, s);
                launch_m2l_block(block_args(P, B, true, P.dL32, P.dL, 0), B.tb, B.grp, 1, s);
            } else if (B.use)
                launch_m2l_block(block_args(P, B, false, P.dL, P.dL, 0), B.tb, B.grp, 0, s);
            else if (P.l2l[L].n_targets)
                launch_xlate(xargs(P, P.l2l[L], P.dL, P.dL, 1), P.l2l[L].n_targets, s);
        }
        mark(5);
        if (field) {
            launch_fill_zero(P.d_far_e, 3 * P.n, s);
            launch_l2p_field(P.d_far_leaves, P.n_far_leaves, bx, lv, P.dX, P.dY, P.dZ, P.dL, P.k, P.p_leafmax,
                             P.d_far, P.d_far_e, s);
        } else {
            for (const auto& r : P.l2p_runs)
                launch_l2p(P.d_leafdesc + r.first, r.n, lv, P.dX, P.dY, P.dZ, P.dL, P.k, r.p, P.d_far, s);
        }
        mark(6);
    }
    if (parts & kSeqP2P) {
        P2PArgs pa = p2p_args(P, out_mode, out);
        pa.far_e = P.d_far_e;
        pa.field = field;
        if (field)
            launch_p2p_field(pa, P.field_items, P.precision, s);
        else
            launch_p2p(pa, P.near_items, P.precision, P.p2p_lowk, P.p2p_tile, s);
        mark(7);
    }
}

// one evaluate into `out` of out_type (HFMM_C64: the FP64 result lands in d_out and is
// rounded into out)
void sequence_typed(hfmm_plan& P, const void* q, int q_type, void* out, int out_type, hipStream_t s) {
    if (out_type == HFMM_C64) {
        run_sequence(P, q, q_type, P.d_out, s, nullptr);
        launch_to_c64(P.d_out, (float2*)out, P.n, s);
    } else {
        run_sequence(P, q, q_type, (double2*)out, s, nullptr);
    }
}

void evaluate_device(hfmm_plan& P, const void* q, int q_type, void* out, hipStream_t s, int out_type = HFMM_C128) {
    alloc_wave_parts(P);
    if (!P.use_graph) {
        sequence_typed(P, q, q_type, out, out_type, s);
        return;
    }
    if (!P.gexec || P.g_q != q || P.g_out != out || P.g_qtype != q_type || P.g_outtype != out_type) {
        if (P.gexec) {
            HIPCHK(hipGraphExecDestroy(P.gexec));
            P.gexec = nullptr;
        }
        if (P.graph) {
            HIPCHK(hipGraphDestroy(P.graph));
            P.graph = nullptr;
        }
        HIPCHK(hipStreamBeginCapture(P.stream, hipStreamCaptureModeThreadLocal));
        try {
            sequence_typed(P, q, q_type, out, out_type, P.stream);
        } catch (...) {
            hipGraph_t g = nullptr;
            (void)hipStreamEndCapture(P.stream, &g);
            if (g) (void)hipGraphDestroy(g);
            throw;
        }
        HIPCHK(hipStreamEndCapture(P.stream, &P.graph));
        HIPCHK(hipGraphInstantiate(&P.gexec, P.graph, nullptr, nullptr, 0));
        P.g_q = q;
        P.g_out = out;
        P.g_qtype = q_type;
        P.g_outtype = out_type;
    }
    HIPCHK(hipGraphLaunch(P.gexec, s));
}

}  // namespace

namespace {
int guard_impl(void (*fn)(void*), void* ctx) {
    try {
        fn(ctx);
        return HFMM_OK;
    } catch (const Error& e) {
        g_last_error = e.msg;
        return e.code;
    } catch (const std::bad_alloc&) {
        g_last_error = "host allocation failed";
        return HFMM_ERR_MEMORY;
    } catch (const std::exception& e) {
        g_last_error = e.what();
        return HFMM_ERR_INTERNAL;
    } catch (...) {
        g_last_error = "unknown error";
        return HFMM_ERR_INTERNAL;
    }
}
template <typename F>
int guarded(F&& f) {
    return guard_impl([](void* c) { (*(F*)c)(); }, (void*)&f);
}
}  // namespace

static void export_tree(const Tree& t, int* level, uint64_t* code, int* count, int* pstart, int* parent,
                        uint8_t* is_leaf, int64_t* perm);
static void export_list(const Lists& ls, char which, int* pairs);

extern "C" {

void hfmm_opts_default(hfmm_opts* o) {
    std::memset(o, 0, sizeof(*o));
    o->p = 4;
    o->n_max = 16;
    o->max_depth = 0;
    o->precision = HFMM_PREC_FP64;
    o->use_graph = 1;
    o->m2l_kernel = 0;
    o->m2l_fp64_levels = -1;
    o->p2p_tile = 0;
}

int hfmm_plan_create(const double* xyz, int64_t n, double k, const hfmm_opts* o, hfmm_plan** out) {
    return guarded([&] {
        if (!out || !o || !xyz) fail(HFMM_ERR_ARG, "null argument");
        *out = nullptr;
        hfmm_plan* P = new hfmm_plan();
        try {
            build_plan(*P, xyz, n, k, *o);
        } catch (...) {
            delete P;
            throw;
        }
        *out = P;
    });
}

int hfmm_plan_info_get(const hfmm_plan* P, hfmm_plan_info* info) {
    return guarded([&] {
        if (!P || !info) fail(HFMM_ERR_ARG, "null argument");
        std::memset(info, 0, sizeof(*info));
        info->n_points = P->n;
        info->depth = P->depth;
        info->n_boxes = P->tree.n_boxes();
        info->n_leaves = P->n_leaves;
        info->n_leaves_phase64 = P->precision == HFMM_PREC_MIXED ? P->n_leaves - P->n_p2p_fp32 : 0;
        info->maxleaf = P->tree.maxleaf;
        info->n_v = (int64_t)P->lists.v_tgt.size();
        info->n_u = (int64_t)P->lists.u_tgt.size();
        info->n_w = (int64_t)P->lists.w_tgt.size();
        info->n_x = (int64_t)P->lists.x_tgt.size();
        info->n_p2p_pairs = P->n_p2p_pairs;
        for (int L = 0; L < HFMM_MAX_LEVELS; ++L) {
            info->p_level[L] = (L >= 1 && L <= P->depth) ? P->p_eff[L] : 0;
            info->p_table[L] = (L >= 1 && L <= P->depth) ? P->p_level[L] : 0;
            if ((P->m2lb[L].use && P->m2lb[L].fp32) || (P->m2lc[L].use && P->m2lc[L].fp32))
                info->m2l_fp32_levels |= 1 << L;
            if (P->m2mb[L].use && P->m2mb[L].fp32) info->m2m_fp32_levels |= 1 << L;
            if (P->l2lb[L].use && P->l2lb[L].fp32) info->l2l_fp32_levels |= 1 << L;
        }
        info->n_leaves_coord32 = P->n_leaves_coord32;
        info->extent = P->tree.extent;
        for (int a = 0; a < 3; ++a) info->pmin[a] = P->tree.pmin[a];
    });
}

int hfmm_plan_wave_levels(const hfmm_plan* P, int* m2l, int* m2m, int* l2l) {
    return guarded([&] {
        if (!P) fail(HFMM_ERR_ARG, "null plan");
        auto mask = [](const M2LWaveLevel* levels, int* out) {
            if (!out) return;
            *out = 0;
            for (int L = 0; L < kMaxLevels; ++L)
                if (levels[L].use) *out |= 1 << L;
        };
        mask(P->m2lc, m2l);
        mask(P->m2mc, m2m);
        mask(P->l2lc, l2l);
    });
}

int hfmm_plan_export_tree(const hfmm_plan* P, int* level, uint64_t* code, int* count, int* pstart, int* parent,
                          uint8_t* is_leaf, int64_t* perm) {
    return guarded([&] {
        if (!P) fail(HFMM_ERR_ARG, "null plan");
        export_tree(P->tree, level, code, count, pstart, parent, is_leaf, perm);
    });
}

int hfmm_plan_export_list(const hfmm_plan* P, char which, int* pairs) {
    return guarded([&] {
        if (!P || !pairs) fail(HFMM_ERR_ARG, "null argument");
        export_list(P->lists, which, pairs);
    });
}

int hfmm_plan_set_degrees(hfmm_plan* P, const int* p_level) {
    return guarded([&] {
        if (!P || !p_level) fail(HFMM_ERR_ARG, "null argument");
        int eff[kMaxLevels];
        for (int L = 0; L < kMaxLevels; ++L) {
            eff[L] = P->p_level[L];
            if (L >= HFMM_MAX_LEVELS || L < 1 || L > P->depth || p_level[L] == 0) continue;
            if (p_level[L] < 2 || p_level[L] > P->p_level[L])
                fail(HFMM_ERR_ARG, "p_level entries must be 0 or in [2, table degree of the level]");
            eff[L] = p_level[L];
        }
        HIPCHK(hipStreamSynchronize(P->stream));
        std::copy(eff, eff + kMaxLevels, P->p_eff);
        ++P->degree_version;
        HIPCHK(hipMemcpy(P->d_plevel, P->p_eff, sizeof(int) * kMaxLevels, hipMemcpyHostToDevice));
        for (int L = 0; L < kMaxLevels; ++L)
            for (M2LWaveLevel* B : {&P->m2lc[L], &P->m2mc[L], &P->l2lc[L]})
                if (B->use) pack_wave_coax(*P, *B);
        if (P->gexec) {
            HIPCHK(hipGraphExecDestroy(P->gexec));
            P->gexec = nullptr;
        }
        if (P->graph) {
            HIPCHK(hipGraphDestroy(P->graph));
            P->graph = nullptr;
        }
        P->g_q = nullptr;
    });
}

int hfmm_evaluate_typed(hfmm_plan* P, const void* q, int q_type, void* out, int out_type, int ptr_kind,
                        void* stream) {
    return guarded([&] {
        if (!P || !q || !out) fail(HFMM_ERR_ARG, "null argument");
        if (q_type < HFMM_F64 || q_type > HFMM_C64) fail(HFMM_ERR_ARG, "unknown charge type");
        if (out_type != HFMM_C128 && out_type != HFMM_C64) fail(HFMM_ERR_ARG, "unknown output type");
        hipStream_t s = stream ? (hipStream_t)stream : P->stream;
        if (ptr_kind == HFMM_HOST) {
            HIPCHK(hipMemcpyAsync(P->d_qin, q, (size_t)P->n * charge_bytes(q_type), hipMemcpyHostToDevice, s));
            if (out_type == HFMM_C64) {
                if (!P->d_out32) P->d_out32 = P->alloc<float2>(P->n);
                evaluate_device(*P, P->d_qin, q_type, P->d_out32, s, HFMM_C64);
                HIPCHK(hipMemcpyAsync(out, P->d_out32, (size_t)P->n * 8, hipMemcpyDeviceToHost, s));
            } else {
                evaluate_device(*P, P->d_qin, q_type, P->d_out, s);
                HIPCHK(hipMemcpyAsync(out, P->d_out, (size_t)P->n * 16, hipMemcpyDeviceToHost, s));
            }
        } else if (ptr_kind == HFMM_DEVICE) {
            evaluate_device(*P, q, q_type, out, s, out_type);
        } else {
            fail(HFMM_ERR_ARG, "unknown pointer kind");
        }
        HIPCHK(hipStreamSynchronize(s));
    });
}

int hfmm_evaluate_field(hfmm_plan* P, const void* q, int q_type, void* phi, void* field, int ptr_kind,
                        void* stream) {
    return guarded([&] {
        if (!P || !q || !phi || !field) fail(HFMM_ERR_ARG, "null argument");
        if (q_type < HFMM_F64 || q_type > HFMM_C64) fail(HFMM_ERR_ARG, "unknown charge type");
        if (P->p_leafmax + 1 > kMaxP) fail(HFMM_ERR_ARG, "the field needs leaf degrees of at most 39");
        hipStream_t s = stream ? (hipStream_t)stream : P->stream;
        if (!P->d_far_e) P->d_far_e = P->alloc<double2>(3 * P->n);
        alloc_wave_parts(*P);
        if (ptr_kind == HFMM_HOST) {
            if (!P->d_field_out) P->d_field_out = P->alloc<double2>(3 * P->n);
            HIPCHK(hipMemcpyAsync(P->d_qin, q, (size_t)P->n * charge_bytes(q_type), hipMemcpyHostToDevice, s));
            run_sequence(*P, P->d_qin, q_type, P->d_out, s, nullptr, nullptr, P->d_field_out);
            HIPCHK(hipMemcpyAsync(phi, P->d_out, (size_t)P->n * 16, hipMemcpyDeviceToHost, s));
            HIPCHK(hipMemcpyAsync(field, P->d_field_out, (size_t)P->n * 48, hipMemcpyDeviceToHost, s));
        } else if (ptr_kind == HFMM_DEVICE) {
            run_sequence(*P, q, q_type, (double2*)phi, s, nullptr, nullptr, (double2*)field);
        } else {
            fail(HFMM_ERR_ARG, "unknown pointer kind");
        }
        HIPCHK(hipStreamSynchronize(s));
    });
}

int hfmm_evaluate(hfmm_plan* P, const void* q, int q_type, void* out, int ptr_kind, void* stream) {
    return hfmm_evaluate_typed(P, q, q_type, out, HFMM_C128, ptr_kind, stream);
}

int hfmm_benchmark(hfmm_plan* P, const void* q_dev, int q_type, void* out_dev, int warmup, int reps,
                   double* median_ms, double* phase_ms) {
    return guarded([&] {
        if (!P || !q_dev || !out_dev || reps < 1) fail(HFMM_ERR_ARG, "bad argument");
        hipStream_t s = P->stream;
        for (int i = 0; i < warmup; ++i) evaluate_device(*P, q_dev, q_type, out_dev, s);
        HIPCHK(hipStreamSynchronize(s));
        std::vector<hipEvent_t> ev(2 * reps);
        for (auto& e : ev) HIPCHK(hipEventCreate(&e));
        for (int i = 0; i < reps; ++i) {
            HIPCHK(hipEventRecord(ev[2 * i], s));
            evaluate_device(*P, q_dev, q_type, out_dev, s);
            HIPCHK(hipEventRecord(ev[2 * i + 1], s));
        }
        HIPCHK(hipStreamSynchronize(s));
        std::vector<double> ms(reps);
        for (int i = 0; i < reps; ++i) {
            float f = 0;
            HIPCHK(hipEventElapsedTime(&f, ev[2 * i], ev[2 * i + 1]));
            ms[i] = f;
        }
        for (auto& e : ev) (void)hipEventDestroy(e);
        std::sort(ms.begin(), ms.end());
        if (median_ms) *median_ms = ms[reps / 2];
        if (phase_ms) {
            hipEvent_t pe[8];
            for (auto& e : pe) HIPCHK(hipEventCreate(&e));
            for (int i = 0; i < 7; ++i) phase_ms[i] = 0.0;
            for (int r = 0; r < reps; ++r) {
                run_sequence(*P, q_dev, q_type, (double2*)out_dev, s, pe);
                HIPCHK(hipStreamSynchronize(s));
                for (int i = 0; i < 7; ++i) {
                    float f = 0;
                    HIPCHK(hipEventElapsedTime(&f, pe[i], pe[i + 1]));
                    phase_ms[i] += f / reps;
                }
            }
            for (auto& e : pe) (void)hipEventDestroy(e);
        }
    });
}

int hfmm_benchmark_m2l_levels(hfmm_plan* P, const void* q_dev, int q_type, void* out_dev, int reps,
                              double* level_ms) {
    return guarded([&] {
        if (!P || !q_dev || !out_dev || !level_ms || reps < 1) fail(HFMM_ERR_ARG, "bad argument");
        hipStream_t s = P->stream;
        alloc_wave_parts(*P);
        std::vector<hipEvent_t> ev(2 * kMaxLevels);
        for (auto& e : ev) HIPCHK(hipEventCreate(&e));
        for (int L = 0; L < HFMM_MAX_LEVELS; ++L) level_ms[L] = 0.0;
        for (int r = 0; r < reps; ++r) {
            run_sequence(*P, q_dev, q_type, (double2*)out_dev, s, nullptr, ev.data());
            HIPCHK(hipStreamSynchronize(s));
            for (int L = 2; L <= P->depth && L < HFMM_MAX_LEVELS; ++L) {
                if (!P->m2l[L].n_targets) continue;
                float f = 0;
                HIPCHK(hipEventElapsedTime(&f, ev[2 * L], ev[2 * L + 1]));
                level_ms[L] += f / reps;
            }
        }
        for (auto& e : ev) (void)hipEventDestroy(e);
    });
}

int hfmm_plan_destroy(hfmm_plan* P) {
    return guarded([&] { delete P; });
}

int hfmm_direct(const double* xyz, int64_t n, const double* q, double k, const int64_t* targets, int64_t nt,
                double* out) {
    return guarded([&] {
        if (!xyz || !q || !out || (nt > 0 && !targets) || n <= 0 || nt < 0) fail(HFMM_ERR_ARG, "bad argument");
        if (!std::isfinite(k)) fail(HFMM_ERR_ARG, "k must be a finite real number");
        check_device();
        std::vector<double> X(n), Y(n), Z(n), tx(nt), ty(nt), tz(nt);
        for (int64_t i = 0; i < n; ++i) {
            X[i] = xyz[3 * i];
            Y[i] = xyz[3 * i + 1];
            Z[i] = xyz[3 * i + 2];
        }
        for (int64_t i = 0; i < nt; ++i) {
            if (targets[i] < 0 || targets[i] >= n) fail(HFMM_ERR_ARG, "target index out of range");
            tx[i] = X[targets[i]];
            ty[i] = Y[targets[i]];
            tz[i] = Z[targets[i]];
        }
        hfmm_plan tmp;   // owns the temporaries
        double* dX = tmp.upload(X);
        double* dY = tmp.upload(Y);
        double* dZ = tmp.upload(Z);
        double* dtx = tmp.upload(tx);
        double* dty = tmp.upload(ty);
        double* dtz = tmp.upload(tz);
        double2* dq = tmp.alloc<double2>(n);
        HIPCHK(hipMemcpy(dq, q, (size_t)n * 16, hipMemcpyHostToDevice));
        double2* dout = tmp.alloc<double2>(nt);
        launch_direct(dX, dY, dZ, dq, n, k, dtx, dty, dtz, nt, dout, nullptr);
        HIPCHK(hipDeviceSynchronize());
        if (nt) HIPCHK(hipMemcpy(out, dout, (size_t)nt * 16, hipMemcpyDeviceToHost));
    });
}

struct hfmm_tree {
    Tree tree;
    Lists lists;
};

int hfmm_tree_create(const double* xyz, int64_t n, int n_max, int max_depth, hfmm_tree** out) {
    return guarded([&] {
        if (!out || !xyz) fail(HFMM_ERR_ARG, "null argument");
        *out = nullptr;
        if (n <= 0 || n > (int64_t)1 << 30) fail(HFMM_ERR_ARG, "positions must be a nonempty finite (N,3) array");
        for (int64_t i = 0; i < 3 * n; ++i)
            if (!std::isfinite(xyz[i])) fail(HFMM_ERR_ARG, "positions must be a nonempty finite (N,3) array");
        if (n_max < 1) fail(HFMM_ERR_ARG, "p must be an integer >=2; N_max must be a positive integer");
        hfmm_tree* T = new hfmm_tree();
        try {
            T->tree = build_tree(xyz, n, n_max, max_depth);
            T->lists = build_lists(T->tree);
        } catch (...) {
            delete T;
            throw;
        }
        *out = T;
    });
}

int hfmm_tree_create_device(const double* xyz, int64_t n, int n_max, int max_depth, hfmm_tree** out) {
    return guarded([&] {
        if (!out || !xyz) fail(HFMM_ERR_ARG, "null argument");
        *out = nullptr;
        if (n <= 0 || n > (int64_t)1 << 30) fail(HFMM_ERR_ARG, "positions must be a nonempty finite (N,3) array");
        for (int64_t i = 0; i < 3 * n; ++i)
            if (!std::isfinite(xyz[i])) fail(HFMM_ERR_ARG, "positions must be a nonempty finite (N,3) array");
        if (n_max < 1) fail(HFMM_ERR_ARG, "p must be an integer >=2; N_max must be a positive integer");
        check_device();
        std::unique_ptr<hfmm_tree> T(new hfmm_tree());
        build_tree_device(xyz, n, n_max, max_depth, T->tree, T->lists);
        *out = T.release();
    });
}

int hfmm_tree_info_get(const hfmm_tree* T, hfmm_plan_info* info) {
    return guarded([&] {
        if (!T || !info) fail(HFMM_ERR_ARG, "null argument");
        std::memset(info, 0, sizeof(*info));
        info->n_points = T->tree.n_points;
        info->depth = T->tree.depth;
        info->n_boxes = T->tree.n_boxes();
        int nl = 0;
        for (auto f : T->tree.is_leaf) nl += f;
        info->n_leaves = nl;
        info->maxleaf = T->tree.maxleaf;
        info->n_v = (int64_t)T->lists.v_tgt.size();
        info->n_u = (int64_t)T->lists.u_tgt.size();
        info->n_w = (int64_t)T->lists.w_tgt.size();
        info->n_x = (int64_t)T->lists.x_tgt.size();
        info->extent = T->tree.extent;
        for (int a = 0; a < 3; ++a) info->pmin[a] = T->tree.pmin[a];
    });
}

static void export_tree(const Tree& t, int* level, uint64_t* code, int* count, int* pstart, int* parent,
                        uint8_t* is_leaf, int64_t* perm) {
    if (level) std::copy(t.level.begin(), t.level.end(), level);
    if (code) std::copy(t.code.begin(), t.code.end(), code);
    if (count) std::copy(t.count.begin(), t.count.end(), count);
    if (pstart) std::copy(t.pstart.begin(), t.pstart.end(), pstart);
    if (parent) std::copy(t.parent.begin(), t.parent.end(), parent);
    if (is_leaf) std::copy(t.is_leaf.begin(), t.is_leaf.end(), is_leaf);
    if (perm) std::copy(t.perm.begin(), t.perm.end(), perm);
}

static void export_list(const Lists& ls, char which, int* pairs) {
    const std::vector<int>*a, *b;
    switch (which) {
        case 'V': a = &ls.v_tgt; b = &ls.v_src; break;
        case 'U': a = &ls.u_tgt; b = &ls.u_src; break;
        case 'W': a = &ls.w_tgt; b = &ls.w_src; break;
        case 'X': a = &ls.x_tgt; b = &ls.x_src; break;
        default: fail(HFMM_ERR_ARG, "list must be one of V, U, W, X");
    }
    for (size_t i = 0; i < a->size(); ++i) {
        pairs[2 * i] = (*a)[i];
        pairs[2 * i + 1] = (*b)[i];
    }
}

int hfmm_tree_export(const hfmm_tree* T, int* level, uint64_t* code, int* count, int* pstart, int* parent,
                     uint8_t* is_leaf, int64_t* perm) {
    return guarded([&] {
        if (!T) fail(HFMM_ERR_ARG, "null tree");
        export_tree(T->tree, level, code, count, pstart, parent, is_leaf, perm);
    });
}

int hfmm_tree_export_list(const hfmm_tree* T, char which, int* pairs) {
    return guarded([&] {
        if (!T || !pairs) fail(HFMM_ERR_ARG, "null argument");
        export_list(T->lists, which, pairs);
    });
}

int hfmm_tree_destroy(hfmm_tree* T) {
    return guarded([&] { delete T; });
}

int hfmm_host_jhat(double x, int p, double* out) {
    return guarded([&] {
        if (!out || p < 0 || p > 4 * kMaxP) fail(HFMM_ERR_ARG, "bad argument");
        jhat_host(x, p, out);
    });
}

int hfmm_host_hhat(double x, int p, double* re, double* im) {
    return guarded([&] {
        if (!re || !im || p < 1 || p > 4 * kMaxP) fail(HFMM_ERR_ARG, "bad argument");
        hhat_host(x, p, re, im);
    });
}

int hfmm_host_rotation(double theta, int p, double* out) {
    return guarded([&] {
        if (!out || p < 0 || p > kMaxP) fail(HFMM_ERR_ARG, "bad argument");
        rotation_table(theta, p, out);
    });
}

int hfmm_host_coax(int kind, double k, double t, double rs, double rt, int ps, int pt, double* out) {
    return guarded([&] {
        if (!out || kind < 0 || kind > 2 || ps < 0 || pt < 0 || ps > kMaxP || pt > kMaxP || !(t > 0) ||
            !(rs > 0) || !(rt > 0) || !(k >= 0))
            fail(HFMM_ERR_ARG, "bad argument");
        const Gaunt G = make_gaunt(std::max(ps, pt));
        coax_table(kind, G, k, t, rs, rt, ps, pt, out);
    });
}

const char* hfmm_last_error(void) { return g_last_error.c_str(); }

}  // extern "C"

// ---------------------------------------------------------------------------------
// Batches of independent problems: one plan per problem; an evaluate forks the
// problems over a few streams (balanced by point count) and joins them, all inside
// one captured hipGraph, so that small problems run side by side on the GPU.
// ---------------------------------------------------------------------------------
struct hfmm_batch {
    std::vector<hfmm_plan*> plans;
    std::vector<std::vector<int>> branch;   // problems per stream, largest first
    std::vector<hipStream_t> streams;
    std::vector<hipEvent_t> join, join2;
    hipEvent_t fork = nullptr, fork2 = nullptr;
    hipStream_t stream = nullptr;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    std::vector<const void*> g_q;
    std::vector<void*> g_out;
    std::vector<unsigned> g_ver;            // degree versions of the plans at capture
    int g_qtype = -1;
    // launches over all problems (rebuilt with the graph): the wave and block M2L, one per
    // kernel instance (the block kernel's are persistent), and the near field
    struct WaveInstance {                   // the wave kernels, one launch per degree
        bool fp32 = false;
        int p = 0, n = 0, n_sums = 0;
        const int2* work = nullptr;
        const int4* sums = nullptr;
        const M2LWaveArgs* args = nullptr;
    };
    std::vector<WaveInstance> wave_inst;
    struct M2LInstance {
        int p = 0, tb = 0, g = 0, fp32 = 0, grid = 0;
        size_t shm = 0;
        WorkQueues q{};
    };
    std::vector<M2LInstance> m2l_inst;
    std::vector<const M2LBlockArgs*> m2l_args;   // device descriptors per instance
    const SdRun* sd_runs[2] = {};           // multipoles in (S, D) form, FP64 and FP32
    const int2* sd_work[2] = {};
    int sd_n[2] = {};
    const P2PArgs* d_p2p_args = nullptr;
    const NearItem* p2p_items[4] = {};     // per near-field leaf class (kP2PClass*)
    const int* p2p_prob[4] = {};
    int p2p_n[4] = {};
    int* d_counters = nullptr;
    int n_counters = 0;
    std::vector<void*> pallocs;             // device buffers of the persistent launches
    void free_persistent() {
        for (void* p : pallocs) (void)hipFree(p);
        pallocs.clear();
        m2l_inst.clear();
        m2l_args.clear();
        wave_inst.clear();
        d_p2p_args = nullptr;
        d_counters = nullptr;
    }
    template <typename T>
    T* alloc(size_t n) {
        void* p = nullptr;
        if (hipMalloc(&p, std::max<size_t>(1, n) * sizeof(T)) != hipSuccess)
            fail(HFMM_ERR_MEMORY, "hipMalloc failed (batch work lists)");
        pallocs.push_back(p);
        return (T*)p;
    }
    template <typename T>
    T* upload(const std::vector<T>& v) {
        T* p = alloc<T>(v.size());
        if (!v.empty()) HIPCHK(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
        return (T*)p;
    }
    ~hfmm_batch() {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        free_persistent();
        for (auto e : join) (void)hipEventDestroy(e);
        for (auto e : join2) (void)hipEventDestroy(e);
        if (fork) (void)hipEventDestroy(fork);
        if (fork2) (void)hipEventDestroy(fork2);
        for (auto st : streams) (void)hipStreamDestroy(st);
        if (stream) (void)hipStreamDestroy(stream);
        for (auto P : plans) delete P;
    }
};

namespace {

constexpr int kBatchStreams = 4;

// Partial sums that a batch holds: a launch leaves up to 0.2 GB of a level (FP32, p = 14, 32 targets a
// block), so 256 mixed problems of 2k to 200k points left 4.8 GB and thousands would not fit.  Every
// further launch ends with a tail of its own: at 1 GiB, 64 such problems (1.2 GB) took two launches and
// 18.5 ms instead of 18.0.
constexpr size_t kBatchPartBytes = (size_t)4 << 30;

// kernel instance of the block M2L (the table-degree range selects KT and MAXU)
int m2l_degree_range(int p) { return p <= 7 ? 0 : p <= 11 ? 1 : p <= 15 ? 2 : p <= 17 ? 3 : p <= 19 ? 4 : 5; }

// queues of a work list: kXcds contiguous ranges of equal length
WorkQueues make_queues(hfmm_batch& B, const std::vector<int2>& work, int* counters) {
    std::vector<int> start(kXcds + 1);
    for (int x = 0; x <= kXcds; ++x) start[x] = (int)((int64_t)work.size() * x / kXcds);
    WorkQueues q;
    q.work = B.upload(work);
    q.start = B.upload(start);
    q.count = counters;
    return q;
}

// Device descriptors and work lists of the launches over all problems for the current
// degrees and pointers: the M2L levels of every problem grouped by kernel instance, and the
// near-field items of every problem.
void build_persistent(hfmm_batch& B, void* const* out, int q_type) {
    B.free_persistent();
    const int np = (int)B.plans.size();
    std::map<std::array<int, 4>, std::vector<M2LBlockArgs>> groups;
    std::map<std::array<int, 4>, int> pmax;
    for (int i = 0; i < np; ++i) {
        hfmm_plan& P = *B.plans[i];
        for (int L = 2; L <= P.depth; ++L) {
            const M2LBlockLevel& lb = P.m2lb[L];
            if (!P.m2l[L].n_targets || !lb.use || lb.n_items <= 0) continue;
            const int pk = std::max(lb.ps, lb.pt);
            const std::array<int, 4> key{m2l_degree_range(pk), lb.tb, lb.grp, lb.fp32 ? 1 : 0};
            groups[key].push_back(block_args(P, lb, lb.fp32, lb.fp32 ? (const void*)P.dM32 : (const void*)P.dM, P.dL, 0));
            pmax[key] = std::max(pmax[key], pk);
        }
    }
    // wave kernel: one launch per degree over problems and levels, split to twice the items
    // of a single level.  Split by level as for a plan alone, 16 problems of 2k to 20k points at
    // p = 10 made 36128 items, of a group or two each: 2.67 ms, and 0.29 for the sums, against
    // 1.37 and 0.05 for the 6016 items of this rule.
    // FP32 levels keep their items: they decide what is summed in FP32, and a batch gives each
    // problem's own result.
    using WaveKey = std::pair<bool, int>;   // FP32, degree
    std::map<WaveKey, std::vector<std::pair<hfmm_plan*, const M2LWaveLevel*>>> waves;
    std::map<WaveKey, int64_t> wave_groups;
    for (int fp32 = 0; fp32 < 2; ++fp32) {
        std::vector<SdRun> runs;
        std::vector<int2> work;
        for (const hfmm_plan* P : B.plans)
            for (const LevelRun& r : sd_runs(*P)) {
                if (r.fp32 != (bool)fp32) continue;
                const int entries = (r.p + 1) * (r.p + 2) / 2;
                const int64_t n = (int64_t)r.n * (fp32 ? (entries + 1) / 2 : entries);
                for (int64_t c = 0; c * kSdChunk < n; ++c) work.push_back(make_int2((int)runs.size(), (int)c));
                runs.push_back({P->dM + P->exp_off[r.b0],
                                fp32 ? (void*)(P->dMs32 + 2 * P->sd32_off[r.b0]) : (void*)(P->dMs + P->sd_off[r.b0]), n,
                                r.p + 1, 0});
            }
        B.sd_n[fp32] = (int)work.size();
        B.sd_runs[fp32] = B.upload(runs);
        B.sd_work[fp32] = B.upload(work);
    }
    for (hfmm_plan* P : B.plans)
        for (const M2LWaveLevel& c : P->m2lc) {
            if (!c.use || !c.n_groups) continue;
            const int pk = std::max(P->p_eff[c.src_level], P->p_eff[c.tgt_level]);
            waves[{c.fp32, pk}].push_back({P, &c});
            wave_groups[{c.fp32, pk}] += c.n_groups;
        }
    B.n_counters = 16 * kXcds * (int)groups.size();
    std::vector<int> zeros(B.n_counters, 0);
    B.d_counters = B.upload(zeros);
    int qi = 0;
    for (auto& kv : groups) {
        hfmm_batch::M2LInstance in;
        in.p = pmax[kv.first];
        in.tb = kv.first[1];
        in.g = kv.first[2];
        in.fp32 = kv.first[3];
        in.shm = m2l_block_lds_bytes(in.p, in.tb, in.g, in.fp32 ? 4 : 8);
        std::vector<int2> work;
        for (int j = 0; j < (int)kv.second.size(); ++j)
            for (int t = 0; t < kv.second[j].n_items; ++t) work.push_back(make_int2(j, t));
        const M2LBlockArgs* d_args = B.upload(kv.second);
        in.q = make_queues(B, work, B.d_counters + 16 * kXcds * qi++);
        in.grid = m2l_block_persistent_grid(in.p, in.tb, in.g, in.fp32, in.shm);
        B.m2l_inst.push_back(in);
        B.m2l_args.push_back(d_args);
    }
    // The launches run one after another and share one buffer of partial sums; a launch takes levels
    // up to kBatchPartBytes of them (or one level that needs more).
    struct Pending {
        hfmm_batch::WaveInstance in;
        std::vector<M2LWaveArgs> args;
        std::vector<size_t> part;               // offset of each descriptor's partial sums
        std::vector<int2> work;
        std::vector<int4> sums;
        size_t bytes = 0;
    };
    std::vector<Pending> launches;
    for (auto& kv : waves) {   // every translation's items are a multiple of kXcds
        const bool fp32 = kv.first.first;
        const int p = kv.first.second;
        const int per_item = (int)std::max<int64_t>(1, (wave_groups[kv.first] + 2 * kWaveItems - 1) / (2 * kWaveItems));
        bool first = true;
        for (auto& [P, c] : kv.second) {
            std::vector<int> part_ptr = c->host_part_ptr;
            M2LWaveArgs w = wave_args(*P, *c, wave_source(*P, *c), P->dL, fp32);
            if (!fp32) {
                const std::vector<int4> items =
                    wave_items(P->tree, c->host_targets, c->host_ptr, c->tb, per_item, part_ptr);
                w.n_items = (int)items.size();
                w.items = B.upload(items);
                w.part_ptr = B.upload(part_ptr);
            }
            const size_t bytes = wave_part_bytes(*c, part_ptr[c->n_blocks]);
            if (first || launches.back().bytes + bytes > kBatchPartBytes) {
                launches.emplace_back();
                launches.back().in.fp32 = fp32;
                launches.back().in.p = p;
                first = false;
            }
            Pending& l = launches.back();
            const int j = (int)l.args.size();
            l.part.push_back(l.bytes);
            l.bytes += bytes;
            w.part = nullptr;
            for (int t = 0; t < w.n_items; ++t) l.work.push_back(make_int2(j, t));
            const int chunks = fp32 ? wave32_sum_chunks(p, c->tb) : wave64_sum_chunks(p, c->tb);
            for (int b = 0; b < c->n_blocks; ++b)
                if (part_ptr[b + 1] > part_ptr[b])
                    for (int i = 0; i < chunks; ++i) l.sums.push_back(make_int4(j, b, i, 0));
            l.args.push_back(w);
        }
    }
    size_t most = 0;
    for (const Pending& l : launches) most = std::max(most, l.bytes);
    char* parts = most ? B.alloc<char>(most) : nullptr;
    for (Pending& l : launches) {
        for (size_t j = 0; j < l.args.size(); ++j)
            if ((j + 1 < l.part.size() ? l.part[j + 1] : l.bytes) > l.part[j]) l.args[j].part = parts + l.part[j];
        l.in.n = (int)l.work.size();
        l.in.work = B.upload(l.work);
        l.in.n_sums = (int)l.sums.size();
        l.in.sums = B.upload(l.sums);
        l.in.args = B.upload(l.args);
        B.wave_inst.push_back(l.in);
    }
    std::vector<P2PArgs> pa(np);
    // leaves [l0, l1) of a problem in near-field class cls
    auto leaves = [](const hfmm_plan& P, int cls) {
        const bool fp64 = P.precision == HFMM_PREC_FP64;
        if (fp64 ? cls != kP2PClassFp64 : P.p2p_lowk ? cls != kP2PClassLowK : cls < kP2PClassPhase32)
            return std::make_pair(0, 0);
        if (fp64 || P.p2p_lowk) return std::make_pair(0, P.n_leaves);
        return cls == kP2PClassPhase32 ? std::make_pair(0, P.n_p2p_fp32) : std::make_pair(P.n_p2p_fp32, P.n_leaves);
    };
    for (int i = 0; i < np; ++i)
        pa[i] = p2p_scaled(p2p_args(*B.plans[i], out_mode_of(*B.plans[i], q_type), (double2*)out[i]),
                           B.plans[i]->precision, B.plans[i]->p2p_lowk);
    B.d_p2p_args = B.upload(pa);
    for (int c = 0; c < 4; ++c) {
        int64_t pairs = 0;
        for (const hfmm_plan* P : B.plans) {
            const auto [l0, l1] = leaves(*P, c);
            pairs += near_pairs(P->leaf_box, P->leaf_total, P->tree, l0, l1);
        }
        NearWork w;
        for (int i = 0; i < np; ++i) {
            const hfmm_plan& P = *B.plans[i];
            const auto [l0, l1] = leaves(P, c);
            // the chunks of a mixed problem are those of its plan alone at the default tile of two
            // targets per lane (other tiles split the sources over the lanes otherwise): they decide
            // which sources are summed in FP32, and a batch gives each problem's own result
            if (c == kP2PClassFp64)
                w.add(P.tree, P.leaf_box, P.leaf_total, l0, l1, kP2PFp64TargetsPerLane, near_limit(pairs), i);
            else
                w.add(P.tree, P.leaf_box, P.leaf_total, l0, l1, kP2PBatchTargetsPerLane,
                      near_limit(near_pairs(P.leaf_box, P.leaf_total, P.tree, l0, l1)), i);
        }
        const auto [items, prob] = w.ordered();
        B.p2p_n[c] = (int)items.size();
        B.p2p_items[c] = B.upload(items);
        B.p2p_prob[c] = B.upload(prob);
    }
}

// ev (optional, 5 events): brackets of the upward part, the M2L, the downward part and the
// near field
void batch_sequence(hfmm_batch& B, const void* const* q, int q_type, void* const* out, hipStream_t s,
                    hipEvent_t* ev = nullptr) {
    auto mark = [&](int i) {
        if (ev) HIPCHK(hipEventRecord(ev[i], s));
    };
    mark(0);
    launch_clear_ints(B.d_counters, B.n_counters, s);
    // upward passes and the generic-kernel M2L levels, problems forked over the streams
    HIPCHK(hipEventRecord(B.fork, s));
    for (size_t b = 0; b < B.streams.size(); ++b) {
        HIPCHK(hipStreamWaitEvent(B.streams[b], B.fork, 0));
        for (int i : B.branch[b])
            run_sequence(*B.plans[i], q[i], q_type, (double2*)out[i], B.streams[b], nullptr, nullptr, nullptr,
                         kSeqUp | kSeqM2LGeneric);
        HIPCHK(hipEventRecord(B.join[b], B.streams[b]));
        HIPCHK(hipStreamWaitEvent(s, B.join[b], 0));
    }
    mark(1);
    // the matrix-core M2L of every problem and level: persistent launches of the block
    // kernel, the wave kernels' items.  The (S, D) form of all problems in one launch: every node of a
    // captured graph costs some 10 us of a batch (64 problems of 30 points at p = 4: 2.2 ms with the block
    // kernel, 2.8 with a conversion per problem).
    launch_to_sd64_batch(B.sd_runs[0], B.sd_work[0], B.sd_n[0], s);
    launch_to_sd32_batch(B.sd_runs[1], B.sd_work[1], B.sd_n[1], s);
    for (size_t j = 0; j < B.m2l_inst.size(); ++j) {
        const auto& in = B.m2l_inst[j];
        launch_m2l_block_persistent(B.m2l_args[j], in.q, in.grid, in.p, in.tb, in.g, in.fp32, in.shm, s);
    }
    for (const auto& in : B.wave_inst) {
        (in.fp32 ? launch_m2l_wave32_batch : launch_m2l_wave64_batch)(in.args, in.work, in.n, in.sums, in.n_sums, in.p, s);
    }
    mark(2);
    // downward passes
    HIPCHK(hipEventRecord(B.fork2, s));
    for (size_t b = 0; b < B.streams.size(); ++b) {
        HIPCHK(hipStreamWaitEvent(B.streams[b], B.fork2, 0));
        for (int i : B.branch[b])
            run_sequence(*B.plans[i], q[i], q_type, (double2*)out[i], B.streams[b], nullptr, nullptr, nullptr, kSeqDown);
        HIPCHK(hipEventRecord(B.join2[b], B.streams[b]));
        HIPCHK(hipStreamWaitEvent(s, B.join2[b], 0));
    }
    mark(3);
    // the near field of every problem: one launch per leaf class
    for (int c = 0; c < 4; ++c) launch_p2p_batch(c, B.d_p2p_args, B.p2p_items[c], B.p2p_prob[c], B.p2p_n[c], s);
    mark(4);
}

void batch_evaluate_device(hfmm_batch& B, const void* const* q, int q_type, void* const* out, hipStream_t s) {
    const size_t np = B.plans.size();
    bool same = B.gexec && B.g_qtype == q_type;
    for (size_t i = 0; same && i < np; ++i)
        same = B.g_q[i] == q[i] && B.g_out[i] == out[i] && B.g_ver[i] == B.plans[i]->degree_version;
    if (!same) {
        if (B.gexec) HIPCHK(hipGraphExecDestroy(B.gexec));
        if (B.graph) HIPCHK(hipGraphDestroy(B.graph));
        B.gexec = nullptr;
        B.graph = nullptr;
        build_persistent(B, out, q_type);
        HIPCHK(hipStreamBeginCapture(B.stream, hipStreamCaptureModeThreadLocal));
        try {
            batch_sequence(B, q, q_type, out, B.stream);
        } catch (...) {
            hipGraph_t g = nullptr;
            (void)hipStreamEndCapture(B.stream, &g);
            if (g) (void)hipGraphDestroy(g);
            throw;
        }
        HIPCHK(hipStreamEndCapture(B.stream, &B.graph));
        HIPCHK(hipGraphInstantiate(&B.gexec, B.graph, nullptr, nullptr, 0));
        B.g_q.assign(q, q + np);
        B.g_out.assign(out, out + np);
        B.g_ver.resize(np);
        for (size_t i = 0; i < np; ++i) B.g_ver[i] = B.plans[i]->degree_version;
        B.g_qtype = q_type;
    }
    HIPCHK(hipGraphLaunch(B.gexec, s));
}

}  // namespace

extern "C" {

int hfmm_batch_create(int n_problems, const double* const* xyz, const int64_t* n, const double* k,
                      const hfmm_opts* opts, hfmm_batch** out) {
    return guarded([&] {
        if (!out || !xyz || !n || !k || !opts || n_problems < 1) fail(HFMM_ERR_ARG, "bad argument");
        *out = nullptr;
        std::unique_ptr<hfmm_batch> B(new hfmm_batch());
        for (int i = 0; i < n_problems; ++i) {
            if (!xyz[i]) fail(HFMM_ERR_ARG, "null positions of problem " + std::to_string(i));
            hfmm_plan* P = new hfmm_plan();
            try {
                P->in_batch = true;
                build_plan(*P, xyz[i], n[i], k[i], opts[i]);
            } catch (const Error& e) {
                delete P;
                fail(e.code, "problem " + std::to_string(i) + ": " + e.msg);
            }
            B->plans.push_back(P);
        }
        const int ns = std::min(kBatchStreams, n_problems);
        B->branch.resize(ns);
        std::vector<int> order(n_problems);
        for (int i = 0; i < n_problems; ++i) order[i] = i;
        std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return n[a] > n[b]; });
        std::vector<int64_t> load(ns, 0);
        for (int i : order) {
            const int b = (int)(std::min_element(load.begin(), load.end()) - load.begin());
            B->branch[b].push_back(i);
            load[b] += n[i];
        }
        HIPCHK(hipStreamCreateWithFlags(&B->stream, hipStreamNonBlocking));
        B->streams.resize(ns);
        B->join.resize(ns);
        B->join2.resize(ns);
        for (int b = 0; b < ns; ++b) {
            HIPCHK(hipStreamCreateWithFlags(&B->streams[b], hipStreamNonBlocking));
            HIPCHK(hipEventCreateWithFlags(&B->join[b], hipEventDisableTiming));
            HIPCHK(hipEventCreateWithFlags(&B->join2[b], hipEventDisableTiming));
        }
        HIPCHK(hipEventCreateWithFlags(&B->fork, hipEventDisableTiming));
        HIPCHK(hipEventCreateWithFlags(&B->fork2, hipEventDisableTiming));
        *out = B.release();
    });
}

int hfmm_batch_plan(hfmm_batch* B, int i, hfmm_plan** plan) {
    return guarded([&] {
        if (!B || !plan || i < 0 || i >= (int)B->plans.size()) fail(HFMM_ERR_ARG, "bad argument");
        *plan = B->plans[i];
    });
}

int hfmm_batch_evaluate(hfmm_batch* B, const void* const* q, int q_type, void* const* out, int ptr_kind,
                        void* stream) {
    return guarded([&] {
        if (!B || !q || !out) fail(HFMM_ERR_ARG, "null argument");
        if (q_type < HFMM_F64 || q_type > HFMM_C64) fail(HFMM_ERR_ARG, "unknown charge type");
        const size_t np = B->plans.size();
        for (size_t i = 0; i < np; ++i)
            if (!q[i] || !out[i]) fail(HFMM_ERR_ARG, "null charges or output of problem " + std::to_string(i));
        hipStream_t s = stream ? (hipStream_t)stream : B->stream;
        if (ptr_kind == HFMM_HOST) {
            std::vector<const void*> qd(np);
            std::vector<void*> od(np);
            for (size_t i = 0; i < np; ++i) {
                hfmm_plan& P = *B->plans[i];
                HIPCHK(hipMemcpyAsync(P.d_qin, q[i], (size_t)P.n * charge_bytes(q_type), hipMemcpyHostToDevice, s));
                qd[i] = P.d_qin;
                od[i] = P.d_out;
            }
            batch_evaluate_device(*B, qd.data(), q_type, od.data(), s);
            for (size_t i = 0; i < np; ++i)
                HIPCHK(hipMemcpyAsync(out[i], B->plans[i]->d_out, (size_t)B->plans[i]->n * 16,
                                      hipMemcpyDeviceToHost, s));
        } else if (ptr_kind == HFMM_DEVICE) {
            batch_evaluate_device(*B, q, q_type, out, s);
        } else {
            fail(HFMM_ERR_ARG, "unknown pointer kind");
        }
        HIPCHK(hipStreamSynchronize(s));
    });
}

int hfmm_batch_benchmark(hfmm_batch* B, const void* const* q_dev, int q_type, void* const* out_dev, int warmup,
                         int reps, double* median_ms) {
    return guarded([&] {
        if (!B || !q_dev || !out_dev || reps < 1 || !median_ms) fail(HFMM_ERR_ARG, "bad argument");
        hipStream_t s = B->stream;
        for (int i = 0; i < warmup; ++i) batch_evaluate_device(*B, q_dev, q_type, out_dev, s);
        HIPCHK(hipStreamSynchronize(s));
        std::vector<hipEvent_t> ev(2 * reps);
        for (auto& e : ev) HIPCHK(hipEventCreate(&e));
        for (int i = 0; i < reps; ++i) {
            HIPCHK(hipEventRecord(ev[2 * i], s));
            batch_evaluate_device(*B, q_dev, q_type, out_dev, s);
            HIPCHK(hipEventRecord(ev[2 * i + 1], s));
        }
        HIPCHK(hipStreamSynchronize(s));
        std::vector<double> ms(reps);
        for (int i = 0; i < reps; ++i) {
            float f = 0;
            HIPCHK(hipEventElapsedTime(&f, ev[2 * i], ev[2 * i + 1]));
            ms[i] = f;
        }
        for (auto& e : ev) (void)hipEventDestroy(e);
        std::sort(ms.begin(), ms.end());
        *median_ms = ms[reps / 2];
    });
}

int hfmm_batch_benchmark_phases(hfmm_batch* B, const void* const* q_dev, int q_type, void* const* out_dev, int reps,
                                double* phase_ms) {
    return guarded([&] {
        if (!B || !q_dev || !out_dev || reps < 1 || !phase_ms) fail(HFMM_ERR_ARG, "bad argument");
        hipStream_t s = B->stream;
        batch_evaluate_device(*B, q_dev, q_type, out_dev, s);   // descriptors for these pointers
        HIPCHK(hipStreamSynchronize(s));
        hipEvent_t ev[5];
        for (auto& e : ev) HIPCHK(hipEventCreate(&e));
        for (int i = 0; i < 4; ++i) phase_ms[i] = 0.0;
        for (int r = 0; r < reps; ++r) {
            batch_sequence(*B, q_dev, q_type, out_dev, s, ev);
            HIPCHK(hipStreamSynchronize(s));
            for (int i = 0; i < 4; ++i) {
                float f = 0;
                HIPCHK(hipEventElapsedTime(&f, ev[i], ev[i + 1]));
                phase_ms[i] += f / reps;
            }
        }
        for (auto& e : ev) (void)hipEventDestroy(e);
    });
}

int hfmm_batch_destroy(hfmm_batch* B) {
    return guarded([&] { delete B; });
}

}  // extern "C"
