// Launchers of the HIP kernels (plain pointers; called from the host plan code).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace hfmm {

// Per-box data, device side (canonical box order).
struct DevBoxes {
    const double* centre;      // 3 per box
    const int* level;
    const int* pstart;
    const int* count;
    const int64_t* exp_off;    // offset (in complex coefficients) of the box's expansion
};

// Per-level data, device side.
struct DevLevels {
    const int* p;              // truncation degree per level
    const double* R;           // expansion radius sqrt(3) h per level
};

// Displacement information for one translation direction.
struct DispInfo {
    int theta;                 // index into the rotation tables
    int dist;                  // index of the distance within a level's coaxial tables
};

// Copies the Legendre recurrence coefficients to constant memory (once per process).
void upload_legendre_coefficients();

void launch_fill_zero(double2* buf, int64_t n, hipStream_t s);
void launch_gather_charges(const void* q, int q_type, const int* perm, int64_t n, int conj, double2* q_sorted,
                           hipStream_t s);

// LDS bytes per staged point of the P2M kernel at degree p
inline size_t p2m_bytes_per_point(int p) {
    const size_t P1 = p + 1;
    return 24 * P1 + 32;
}
// points staged per pass of the P2M kernel at the largest leaf degree pmax: the staged
// points and the recurrence coefficients stay within the LDS budget of its workgroup size
int p2m_chunk(int pmax);
// One leaf of the P2M and L2P launches, 64 bytes, read by 16 lanes with one vector load.
struct LeafDesc {
    int box, level, pstart, count;
    int64_t exp_off;           // offset of the leaf's expansion
    int64_t pad0;
    double cx, cy, cz;         // box centre
    double pad1;
};
static_assert(sizeof(LeafDesc) == 64, "LeafDesc is 16 words");

// P2M and L2P run as persistent launches: a grid of resident workgroups, each taking the
// leaves of a contiguous range on its XCD in turn (pmax: the largest leaf degree).
void launch_p2m(const LeafDesc* leaves, int n_items, int chunk, DevLevels lv, const double* X, const double* Y,
                const double* Z, const double2* q, double k, int pmax, double2* M, hipStream_t s);

void launch_l2p(const LeafDesc* leaves, int n_items, DevLevels lv, const double* X, const double* Y, const double* Z,
                const double2* L, double k, int pmax, double2* far, hipStream_t s);

// Generic rotate / coaxial / rotate-back translation over a CSR pair list.
// Target t = targets[blockIdx.x]; sources src[ptr[t_i] .. ptr[t_i+1]) with direction dir[].
// dst[exp_off[t]] (+)= sum over sources of the translated expansion.
struct XlateArgs {
    const int* targets;        // n_targets box ids
    const int* ptr;            // CSR offsets indexed by target ordinal
    const int* src;            // source box ids
    const unsigned short* dir; // direction index per entry
    const DispInfo* dinfo;     // per direction
    const double2* phase;      // per direction, e^{i m phi}, m = 0..pmax
    const double* rot;         // rotation tables, rot_size(pmax) doubles per theta index
    const double2* coax;       // coaxial tables of this launch, indexed by dinfo.dist
    int64_t coax_stride;       // complex entries per coaxial table
    int ps, pt, pmax;          // effective source / target degrees (<= table degrees)
    int tps, tpt;              // degrees the coaxial tables were built for
    int accumulate;            // 1: dst += result, 0: dst = result
    int split;                 // workgroups per target (> 1: contiguous parts of the source
                               // list, added atomically; needs accumulate = 1)
    const double2* srcbuf;
    double2* dstbuf;
    const int64_t* exp_off;
};
void launch_xlate(const XlateArgs& a, int n_targets, hipStream_t s);

// the field E = -grad phi (3 complex values per point, sorted order for far_e, input
// order for field) beside the potential
void launch_l2p_field(const int* leaves, int n_items, DevBoxes bx, DevLevels lv, const double* X, const double* Y,
                      const double* Z, const double2* L, double k, int pmax, double2* far, double2* far_e,
                      hipStream_t s);
// Near field (nearfield.hip) over work items, coordinate differences and r^2 in FP64.
// FP32 (precision != 0): FP32 weights; the items of the first list with an FP32 phase k r, those
// of the second with the phase in FP64 (their pairs reach k r > kP2PFp32MaxKr).  FP64: every leaf
// in FP64 (first list).  Pairs with r^2 <= floor2[leaf] (the coincidence floor of the leaf's
// pairs, in unscaled coordinates) contribute nothing.
constexpr double kP2PFp32MaxKr = 8.0;
// Largest k r over a plan's near pairs for which the mixed near field takes e^{ikr} as
// 1 + ikr (relative error (kr)^2 / 2 <= 5e-9, below FP32 rounding).
constexpr double kP2PLowKr = 1e-4;
// waves that share a work item's sources
constexpr int kNearWaves = 4;
struct NearItem {                 // targets [target, target + n_targets) of a leaf (0: padding)
    int leaf, box, target, n_targets;
};
struct NearItems {
    const NearItem* items = nullptr;
    int n = 0;                    // a multiple of kXcds
};
struct NearBatch {                // 64 consecutive sources of a leaf's ranges
    unsigned long long mask;      // bit i > 0: source i is the first of a range
    int first;                    // range of source 0
    int pad;
};
struct P2PArgs {
    const int* leaf_box;          // leaf -> box
    DevBoxes bx;
    const int* batch_ptr;         // per leaf: its first batch of 64 sources
    const NearBatch* batches;
    const int* rng_delta;         // per range: point of a source minus its number in the leaf
    const int* leaf_src_total;    // sources of each leaf
    const double* floor2;         // per leaf: coincidence floor on r^2 (unscaled coordinates)
    const double *X, *Y, *Z;      // sorted points (FP64)
    const double2* q;             // sorted charges (complex FP64)
    double k;                     // |k|
    double kp_hi, kp_lo;          // |k| / pi in two terms (FP64 near field)
    double scale;                 // coordinate scale of the mixed kernel (set by the launcher)
    double wscale;                // factor of the sums (set by the launcher)
    const double2* far;           // far field per sorted point
    const double2* far_e;         // field: 3 values per sorted point
    const int* perm;              // sorted -> input order
    int out_mode;                 // bit 0: conjugate, bit 1: zero imaginary part
    double2* out;                 // input order
    double2* field;               // 3 values per point, input order
    const unsigned char* coord32; // per leaf (mixed form, FP32 phase): 1 = coordinate differences
                                  // and r^2 in FP32 (null: FP64 at every leaf)
};
constexpr int kP2PFp64TargetsPerLane = 2;   // FP64 near field: two independent chains per lane
constexpr int kP2PFieldTargetsPerLane = 1;
// lowk: every near pair of the plan has k r <= kP2PLowKr (mixed form only); tile: targets
// per lane of the mixed form (1, 2 or 4); items: the two lists
void launch_p2p(const P2PArgs& a, const NearItems* items, int precision, bool lowk, int tile, hipStream_t s);
// the potential and E = -grad phi (a.far_e, a.field set)
void launch_p2p_field(const P2PArgs& a, const NearItems* items, int precision, hipStream_t s);
// Per leaf l < n (leaf order of a): flag[l] = 1 where FP32 coordinates keep the estimated
// relative near-field error of every target of the leaf at or below tol:
//   2^-21 c_max sqrt(sum_j r_j^-4 / sum_j r_j^-2)  <= tol,
// c_max the largest coordinate magnitude relative to the leaf centre over its targets and
// sources (2^-21 c_max bounds the error of an FP32 coordinate difference), the sums over the
// target's sources beyond the coincidence floor (the rounding error of pair j perturbs its
// weight by about r_j^-2 times that error; with random charges the perturbations add in
// quadrature against a potential of about sqrt(sum r_j^-2)).  FP64 arithmetic; setup only.
void launch_p2p_coord_check(const P2PArgs& a, int n, double tol, unsigned char* flag, hipStream_t s);

void launch_direct(const double* X, const double* Y, const double* Z, const double2* q, int64_t n, double k,
                   const double* tx, const double* ty, const double* tz, int64_t nt, double2* out, hipStream_t s);

// M2L on matrix cores over target blocks (m2l_mfma.hip).  The operator tables are
// stored as MFMA A fragments: for a tile (row tile mt, k group kg of four 4-wide
// k-steps) lane l holds, as four consecutive values j = 0..3,
// A[16 mt + l % 16][16 kg + 4 j + l / 16], zero outside the block.
//
// Rotations act on each degree block in the basis u_m = x_m + (-1)^m x_{-m} (m >= 1),
// u_0 = x_0, v_m = x_m - (-1)^m x_{-m} (m >= 1): the reflection x_m -> (-1)^m x_{-m}
// commutes with the rotation exp(-theta G) (G the tridiagonal generator, whose entries are
// symmetric under m -> -m-1), so E_n splits into an (n+1) x (n+1) block on the u and an
// n x n block on the v.  In the LDS buffer u_m sits in the row of x_m and v_m in the row of
// x_{-m}: the u block of degree n is rows n^2+n .. n^2+2n (m ascending), the v block rows
// n^2 .. n^2+n-1 (m = n down to 1).
constexpr int kM2LBlockMaxP = 23;  // largest degree handled by the block kernel
// FP32 one-tile instances: blocks of at most this many rows (forward rotation) or of at
// most this size squared (coaxial) run on the 4x4x1 MFMA in 4-row tiles.  The fragments
// beyond a block's first are loaded when used; with 8 (two tiles) those loads cost more
// than the MFMA passes saved (level-5 M2L at p = 11: 4.38 against 3.90 ms).
constexpr int kM2LQuadMaxRows = 4;
constexpr int kXcds = 8;            // accelerator dies; workgroups are dealt to them round-robin

// Work queues of a persistent launch (batches of problems): work items [start[x],
// start[x+1]) form queue x, one per XCD, each in spatial order; count[16 x] is the next
// index of queue x (one 64-byte line per queue), cleared before every launch.
struct WorkQueues {
    const int2* work;             // (descriptor, item) pairs
    const int* start;             // kXcds + 1 entries
    int* count;                   // 16 kXcds ints
};
#ifdef __HIP__
// The next work item for a workgroup on XCD `home`: its own queue first, then the others'
// (so that the last items are shared out); -1 when every queue is empty.  Indices only
// grow, so every caller returns after at most one pass over the queues.
__device__ inline int work_dequeue(const WorkQueues& q, int home) {
    for (int t = 0; t < kXcds; ++t) {
        const int x = (home + t) % kXcds;
        const int n = q.start[x + 1] - q.start[x];
        int* c = q.count + 16 * x;
        if (__hip_atomic_load(c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= n) continue;
        const int i = atomicAdd(c, 1);
        if (i < n) return q.start[x] + i;
    }
    return -1;
}
#endif
void launch_clear_ints(int* p, int n, hipStream_t s);
constexpr int kM2LMaxAccRegs = 128; // VGPRs per lane for the stage-3 accumulators (block-size choice)
__host__ __device__ constexpr int m2l_tiles(int len) { return (len + 15) / 16; }
// stage-3 units per wave the M2L block kernel is instantiated for at table degree p: the
// units (n, row tile of the n+1 orders), sum_{n<=p} m2l_tiles(n+1), dealt to 4 waves
__host__ __device__ constexpr int m2l_block_maxu(int p) {
    return p <= 7 ? 2 : p <= 11 ? 3 : p <= 15 ? 4 : p <= 17 ? 5 : p <= 19 ? 6 : 8;
}
// FP32 one-tile instances (p <= 15) pack the stage-3 units of the degrees n1 < n2 with
// n1 + n2 = min(p_tab, kM2LPackMax) into one 16-row tile: rows 0..7 take the orders of n1,
// rows 8..15 those of n2 (unit code 256 | n1 << 4 | n2; an odd count leaves the middle
// degree alone), which lowers the units per wave to these
constexpr int kM2LPackMax = 7;
__host__ __device__ constexpr int m2l_block_maxu_packed(int p) { return p <= 7 ? 1 : p <= 11 ? 2 : 3; }
// accumulator VGPRs of a (MAXU units per wave, TB targets, element size) configuration:
// two (u and v) 16x16 tiles per unit and direction column tile
__host__ __device__ constexpr int m2l_acc_regs(int maxu, int tb, int elem_bytes) {
    return maxu * 2 * (2 * tb / 16) * 4 * (elem_bytes / 4);
}
// LDS rows of the expansion block: (p+1)^2 expansion rows, a scratch row that receives
// the stores of rows outside a block, a zero row (read for orders beyond the evaluated
// degree), and as many further zero rows as the padded tiles of the last u block read:
// those reads end at row p^2 + p + 16 m2l_tiles(p+1) - 1.  (At p = 11 in FP32 with 16 x 2
// pairs per group: 148 rows, 38.5 KB, four workgroups per CU.)
__host__ __device__ constexpr int m2l_lds_x_rows(int p) {
    return (p + 1) * (p + 1) + 2 > p * p + p + 16 * m2l_tiles(p + 1) ? (p + 1) * (p + 1) + 2
                                                                      : p * p + p + 16 * m2l_tiles(p + 1);
}
// phase table of the M2L block kernel: entries per (lane parity, direction) for the
// orders m = 0 .. 16 KT - 1 (KT = m2l_tiles(p + 1))
__host__ __device__ constexpr int m2l_phase_len(int p) { return 16 * m2l_tiles(p + 1); }
__host__ __device__ constexpr int m2l_lds_x_elems(int p, int ncol) {
    return (m2l_lds_x_rows(p) * (ncol + 1) + 3) & ~3;
}
struct M2LBlockArgs {
    int p;                           // effective source degree (<= p_tab)
    int p_tab;                       // source degree the tables were built for
    int pt;                          // effective target degree (<= pt_tab); = p for M2L
    int pt_tab;                      // target degree the tables were built for
    int overwrite;                   // store instead of add (every block in one item)
    int n_items;
    const int4* items;               // (block, first group, end group, atomic add)
    const int* blk_targets;          // blocks x TB target boxes (-1: empty slot)
    const unsigned short* grp_dir;   // per group: G directions of equal theta and |d| (0xFFFF: none)
    const int* grp_off;              // per group: G x TB source expansion offsets (-1: none)
    const int* units1;               // forward rotation units: n | block << 8 (0: u, 1: v)
    int n_units1;
    const int* units2;               // coaxial units: |m| (orders +|m| and -|m|)
    int n_units2;
    const int* units3;               // back rotation units: n | row tile << 8 (u and v)
    int n_units3;
    const void* rot1;                // per rotation: fragments of the u and v blocks of E_n^T (T)
    const void* rot3;                // per rotation: fragments of the u and v blocks of E_n (T)
    const int* rot_off1;             // offsets of (n, block) [2 n + block] within rot1's rotation
    const int* rot_off1q;            // blocks of at most 4 rows: their 4x4x1 fragments (-1: larger)
    const int* rot_off3;             // the same within rot3's
    const int* rot_off3p;            // packed stage-3 units (n1, n2): [8 n1 + n2] within rot3's
    int rot_stride1, rot_stride3;
    const void* phase;               // e^{i m phi} per direction (T complex)
    int phase_stride;
    const DispInfo* dinfo;
    const void* coax;                // per distance: fragments of T^m, re then im per lane (T)
    const int* coax_off;             // offset of order m's fragments within one distance
    const int* coax_offq;            // blocks of at most 4 x 4: their 4x4x1 fragments (-1: larger)
    int coax_stride;
    const void* M;                   // multipoles (T complex)
    double2* L;                      // local expansions (FP64), accumulated into
    const int64_t* exp_off;
};
size_t m2l_block_lds_bytes(int p, int tb, int g, int precision_bytes);
void prepare_m2l_block(int p, int tb, int g, int fp32);
void launch_m2l_block(const M2LBlockArgs& a, int tb, int g, int fp32, hipStream_t s);
// Persistent form over many translations (batches): the resident grid of the instance for
// (p = larger table degree, tb, g, fp32) with `shm` bytes of LDS, and the launch over the
// device descriptors d_args and the queues q of (descriptor, item) work.
int m2l_block_persistent_grid(int p, int tb, int g, int fp32, size_t shm);
// FP64 translations with one wave per work item (m2l_wave64.hip).  Operators are stored as MFMA
// A fragments: element (row i, column k) of a block sits in register k / 4, lane 16 (k % 4) + i.
// Rotations, per theta: for n = 0, 1, ... the u block ((n+1) x (n+1)), then the v block (rows
// m = 1..n in the forward table; rows m = 0..n, the first zero, in the back table; columns
// m = 1..n), two registers per lane side by side.  Coaxial tables, per distance: for m = 0..P
// registers m / 4 .. P / 4 (rows and columns are degrees), Re and Im per lane side by side.
constexpr int kWave64MaxP = 14;
constexpr int kWave64Pairs = 16;              // pairs per group
// accumulator registers (four orders each) of degrees 0..p
__host__ __device__ constexpr int wave64_regs(int p) {
    int k = 0;
    for (int n = 0; n <= p; ++n) k += n / 4 + 1;
    return k;
}
__host__ __device__ constexpr int wave64_rot_regs(int n, int h) {   // register pairs before (n, h)
    return 2 * n + (n > 8 ? n - 8 : 0) + (n > 9 ? n - 9 : 0) + (h ? (n >= 8 ? 2 : 1) : 0);
}
__host__ __device__ constexpr int wave64_coax_regs(int P, int m) {   // registers before order m
    return m * (P / 4 + 1) - (4 * ((m / 4) * (m / 4 - 1) / 2) + (m % 4) * (m / 4));
}
// (S, D) buffers start with a block of zeros, the source of absent pairs, and end with padding
// that the last box's gather may read past its entries
__host__ __device__ constexpr int wave_sd_pad(int pmax) { return (pmax + 1) * (pmax + 2) / 2 + 8; }
struct M2LWaveArgs {
    int ps, pt;                      // effective source and target degrees
    int overwrite;                   // store instead of add: targets that this launch alone writes
    int n_items;
    const int4* items;               // (block, first group, end group, part): part 0 is the whole
                                     // block, s > 0 leaves its sums in slot s - 1 of `part`
    int n_blocks;
    void* part;                      // partial sums of split blocks (null: none); FP64: per slot
                                     // and accumulator register 4 tb double4, FP32: per slot the
                                     // U, then the V entries, 2 tb floats each
    const int* part_ptr;             // n_blocks + 1: the slots of each block
    int tb;                          // targets per block, a power of two up to the pairs per group
    const int* blk_targets;          // blocks x tb target boxes (-1: empty slot)
    const int* grp_class;            // per group: theta | dist << 16
    const int* grp_src;              // per pair of a group: source offset in (S, D) entries (no
                                     // pair: 0, a block of zeros)
    const unsigned short* grp_dir;   // per pair: direction
    const void* rot1;                // fragments of E_n^T per theta (forward)
    const void* rot3;                // fragments of E_n per theta (back)
    int rot_stride;
    const void* phase;               // e^{i m phi} per direction
    int phase_stride;
    const void* coax;
    int coax_stride;
    const void* M;                   // (S, D) entries
    double2* L;                      // target expansions (x basis)
    const int64_t* exp_off;
};
void launch_m2l_wave64(const M2LWaveArgs& a, int p, hipStream_t s);
// workgroups that add the parts of one split block of tb targets
int wave64_sum_chunks(int p, int tb);
// many translations of degree p: work[i] = (descriptor, item), n a multiple of kXcds; sums[i] =
// (descriptor, split block, chunk, 0)
void launch_m2l_wave64_batch(const M2LWaveArgs* d_args, const int2* work, int n, const int4* sums, int n_sums, int p,
                             hipStream_t s);
// the expansions of n_boxes consecutive boxes of degree p as (S_re, S_im, D_re, D_im) entries
void launch_to_sd64(const double2* x, double4* sd, int64_t n_boxes, int p, hipStream_t s);

// the same for runs of boxes of many plans: n entries (FP64) or pairs (FP32) of a run, work[i] = (run, chunk)
struct SdRun {
    const double2* x;
    void* sd;
    int64_t n;
    int P1, pad;
};
constexpr int kSdChunk = 1024;
void launch_to_sd64_batch(const SdRun* runs, const int2* work, int n, hipStream_t s);
void launch_to_sd32_batch(const SdRun* runs, const int2* work, int n, hipStream_t s);

// FP32 M2L with one wave per work item (m2l_wave32.hip), the lists as for FP64 with 32 pairs per
// group and source offsets in pairs of (S, D) entries.  M2L alone: source and target degree are the
// same, and the sums are stored (overwrite = 1), the first that a level's locals receive.  The operators are sequences of columns of four
// rows (64 of them per 1 KiB block: wave32_pos).  Rotations, degrees from 1 ascending: split, for the u
// half and from block kWave32VBlock for the v half, per input the output rows; joint, per input k the
// u rows, then (k > 0) the v rows.  Coaxial operators, orders ascending: per input degree the real,
// then the imaginary parts.
constexpr int kWave32MaxP = 15;
constexpr int kWave32Pairs = 32;
// waves per SIMD: two (split layout) while the accumulators leave room in 256 registers, one (joint) above
__host__ __device__ constexpr int wave32_wpe(int p) { return p <= 11 ? 2 : 1; }
__host__ __device__ constexpr int wave32_rot_vecs(int h, int n) {   // columns of degrees below n of half h
    int v = 0;
    for (int j = 1; j < n; ++j) v += (j + 4 - h) / 4 * (j + 1 - h);
    return v;
}
__host__ __device__ constexpr int wave32_joint_vecs(int n) { return wave32_rot_vecs(0, n) + wave32_rot_vecs(1, n); }
__host__ __device__ constexpr int wave32_blocks(int vecs) { return (vecs + 63) / 64; }
constexpr int kWave32VBlock = wave32_blocks(wave32_rot_vecs(0, kWave32MaxP + 1));   // first block of the v rotations
// a theta's rotations: the split layout, then the joint one
constexpr int kWave32SplitFloats = 256 * (kWave32VBlock + wave32_blocks(wave32_rot_vecs(1, kWave32MaxP + 1)));
constexpr int kWave32RotFloats = kWave32SplitFloats + 256 * wave32_blocks(wave32_joint_vecs(kWave32MaxP + 1));
__host__ __device__ constexpr int wave32_coax_vecs(int p, int m) {   // columns of orders below m
    int v = 0;
    for (int j = 0; j < m; ++j) v += 2 * ((p + 1 - j + 3) / 4) * (p + 1 - j);
    return v;
}
constexpr int wave32_pos(int v, int i) { return ((v / 64) * 64 + 4 * (v % 16) + i) * 4 + v % 64 / 16; }   // row i of column v
// pairs of the block of zeros at the front, the source of absent pairs
constexpr int wave32_sd_pad(int pmax) { return (pmax + 1) * (pmax + 2) / 4 + 8; }
void launch_m2l_wave32(const M2LWaveArgs& a, int p, hipStream_t s);
int wave32_sum_chunks(int p, int tb);
void launch_m2l_wave32_batch(const M2LWaveArgs* d_args, const int2* work, int n, const int4* sums, int n_sums, int p,
                             hipStream_t s);
// the expansions of n_boxes consecutive boxes of degree p as FP32 pairs of entries
void launch_to_sd32(const double2* x, float4* sd, int64_t n_boxes, int p, hipStream_t s);

// near field of the problems of a batch: one launch per leaf class (FP64 plans; mixed plans with
// k r <= kP2PLowKr; mixed, FP32 phase; mixed, FP64 phase) over items of all problems,
// d_args[prob[i]] with scale and wscale set (p2p_scaled)
constexpr int kP2PBatchTargetsPerLane = 2;
constexpr int kP2PClassFp64 = 0, kP2PClassLowK = 1, kP2PClassPhase32 = 2, kP2PClassPhase64 = 3;
P2PArgs p2p_scaled(P2PArgs a, int precision, bool lowk);
void launch_p2p_batch(int cls, const P2PArgs* d_args, const NearItem* items, const int* prob, int n, hipStream_t s);
void launch_m2l_block_persistent(const M2LBlockArgs* d_args, const WorkQueues& q, int grid, int p, int tb, int g,
                                 int fp32, size_t shm, hipStream_t s);
void launch_to_float(const double2* in, float2* out, int64_t n, hipStream_t s);
// zero the first ncoef coefficients of the expansions of the given boxes
void launch_zero_boxes(const int* boxes, int n, const int64_t* exp_off, int ncoef, double2* E, hipStream_t s);
// the result rounded to complex64 (output opt-in)
void launch_to_c64(const double2* in, float2* out, int64_t n, hipStream_t s);

}  // namespace hfmm
