// fss_internal.h -- context layout and kernel entry points shared by the
// libfss translation units.  Not part of the public ABI (include/fss.h).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/fss.h"

struct fss_ctx;

// Largest supported interpolation degree and proxy count (p = (d+1)(d+2)/2).
#define FSS_MAX_DEGREE 8
#define FSS_MAX_P 45

namespace fss {

// Thread-local last error message for fss_last_error().
void set_error(const std::string &msg);

#define FSS_HIP(call)                                                                   \
    do {                                                                                \
        hipError_t e_ = (call);                                                         \
        if (e_ != hipSuccess) {                                                         \
            ::fss::set_error(std::string(#call) + ": " + hipGetErrorString(e_));       \
            return FSS_ERR_HIP;                                                         \
        }                                                                               \
    } while (0)

#define FSS_TRY(call)                                                                   \
    do {                                                                                \
        fss_status s_ = (call);                                                         \
        if (s_ != FSS_OK) return s_;                                                    \
    } while (0)

// Count of device-buffer (re)allocations and frees in this process.  A
// captured graph holds raw workspace addresses: it is valid only while this
// count is unchanged since its capture.
uint64_t alloc_epoch();

// Growable device buffer (move-only, freed on destruction).
struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
    DevBuf() = default;
    DevBuf(const DevBuf &) = delete;
    DevBuf &operator=(const DevBuf &) = delete;
    DevBuf(DevBuf &&o) noexcept : p(o.p), bytes(o.bytes) { o.p = nullptr; o.bytes = 0; }
    DevBuf &operator=(DevBuf &&o) noexcept
    {
        if (this != &o) {
            release();
            p = o.p;
            bytes = o.bytes;
            o.p = nullptr;
            o.bytes = 0;
        }
        return *this;
    }
    ~DevBuf() { release(); }
    // grows (contents are not preserved) so that at least nbytes are usable
    fss_status ensure(size_t nbytes);
    void release();
    template <class T> T *as() const { return static_cast<T *>(p); }
};

// Source records (per stage): [0, p0) particle records in tree order, then
// the p proxies of every node at p0 + node * p.
//   Tree order: every particle has one "main" record.  Main records are
//   sorted by the particle's path from level 0 down to the first level where
//   it is not on a node list (then by id), so the main members of any node
//   at any level are one contiguous range.  A particle that the reference's
//   point location drops at some level and finds again deeper (parity
//   assignment, icos_utils.h:139-140) is a member of deeper nodes outside
//   that nesting: each such membership gets an extra "exception" record
//   after the main records, grouped by node.  A node's list is its main
//   range plus its (almost always empty) exception range.
//   Mixed precision: a particle record holds the FP32 offset from the centre
//   of its record node (the deepest node of its main path, or the node of an
//   exception record); a proxy record the offset from its node's centre.

// One work item of the direct-target ("near") kernel: up to 64 targets of one
// node and the list of its class-A source ranges.
struct NearItem {
    int32_t tgt_start; // position of the first target record
    int32_t tgt_cnt;   // 1..64
    int32_t a_beg;     // [a_beg, a_end) into the sorted range list of class A
    int32_t a_end;
    int32_t node;      // global index of the target node
    int32_t out_base;  // output slot of the first target
    int64_t src_off;   // this item's source list in Tree::near_src (set by plan_finish)
    int32_t n_other;   // sources of ranges that cannot hold a target, listed first
    int32_t n_self;    // sources of self ranges, listed after them
};

// A source range: records [start, start + count), all members (or the
// proxies) of node `node`.
struct Range {
    int32_t start;
    int32_t count; // may carry FSS_SELF_BIT
    int32_t node;
    int32_t pad;
};

// One work item of the proxy kernel: the p proxies of one node against one
// chunk of that node's class-B source ranges (long lists are split so that
// every item carries a bounded amount of work).
struct ProxyItem {
    int32_t node;
    int32_t b_beg; // [b_beg, b_end) into the sorted range list of class B
    int32_t b_end;
    int32_t slot; // interpolant slot of the node
};

// The chunks [part_beg, part_end) of one node's proxy work, summed in order
// before the interpolant is solved.
struct ProxySlot {
    int32_t node;
    int32_t part_beg;
    int32_t part_end;
    int32_t pad;
};

// A source range (start, count) whose count carries this bit when the source
// node contains the target node (ancestor or self): the self pair must be
// skipped there (rhs_eval.h:20, fast_rhs.h:107).
#define FSS_SELF_BIT (1 << 30)
// Sources per proxy work item before a node's class-B list is split.
#define FSS_PROXY_CHUNK 4096
// Records per (one-wave) item of the upward pass.
#define FSS_UP_CHUNK 512

// One problem instance of a (possibly batched) tree: particles
// [pbase, pbase + n) of the concatenated state, L levels, and the offset of its
// [L][n] blocks in nodeof / inv_active.
struct Instance {
    int64_t pbase;
    int64_t n;
    int64_t loff;
    int32_t L;
    int32_t pad;
    int64_t rbase; // first source record of the instance (main records first)
    int64_t nbase; // first global node of the instance
};

// Interpolation constants (host copy + device copy).
struct Interp {
    int degree = 2, p = 6;
    std::vector<double> pts;  // p x 3 barycentric nodes
    std::vector<double> lu;   // p x p column-major LU of the Vandermonde
    std::vector<int32_t> ipiv;
    std::vector<double> vinv; // p x p column-major inverse Vandermonde
};

struct Tree {
    bool built = false;
    int L = 0;            // tree levels used (0..L-1)
    int64_t n = 0;        // particles
    int64_t nn = 0;       // nodes on levels 0..L-1
    int64_t ntri_all = 0; // triangles on levels 0..L (geometry is built one level deeper)
    int64_t p0 = 0;       // particle records: n main + exception records
    int64_t nlist = 0;    // sum of the node list lengths (reference lists, export)
    // triangles of levels 0..L and inverse vertex matrices: the context's Geo, or
    // a batch's own arrays below
    const double *d_xyz = nullptr, *d_info = nullptr, *d_tinv = nullptr;
    int64_t nslot_out = 0; // output slots of the near kernel (targets x levels with work)
    int64_t ninter = 0;
    int ngen = 0;
    std::vector<int64_t> level_base; // L+1 entries, host copy
    fss_tree_stats stats{};

    DevBuf tri_xyz, tri_info, tinv; // of a batch, all nodes of all instances (see Geo)
    DevBuf loc;      // int32 [L][n]
    DevBuf found;    // uint8 [L][n]
    DevBuf counts;   // int32 [nn]
    DevBuf inter;    // int32 [7][ninter] AoS
    DevBuf recid;    // int32 [p0]: particle of every record
    DevBuf recnode;  // int32 [p0]: node whose centre is the origin of the record (mixed precision)
    DevBuf rinfo;    // uint8 [p0]: main records: levels on the main path | 0x80 if exception members exist
    DevBuf ipos;     // int32 [n]: main record of every particle
    DevBuf oslot;    // int32 [nn]: output slot of a node's first main target, or -1 (no near work)
    DevBuf nrange;   // int4 [nn]: {main start, main count, exception start, exception count}
    // for memberships outside the main paths (only where there are any: p0 > n)
    DevBuf inv_active; // int32 [L][n]: output slot of a particle in a class-A node, or -1
    DevBuf nodeof;     // int32 [L][n]: global node of a particle per level, or -1 (dropped)
    DevBuf node_slot;  // int32 [nn]: interpolant slot of a node with class-B work, or -1

    // evaluation plan
    int64_t n_near = 0, n_proxy = 0, n_slot = 0, n_ra = 0, n_rb = 0, n_charge = 0;
    DevBuf near_items;  // NearItem[n_near]
    DevBuf near_src;    // int32 source record positions of every near item, item by item
    int64_t n_near_src = 0, n_far_src = 0; // entries of near_src and far_src
    DevBuf proxy_items; // ProxyItem[n_proxy]
    DevBuf proxy_slots; // ProxySlot[n_slot]
    DevBuf far_off;     // int64 [n_proxy + 1]: source list of every proxy item in far_src
    DevBuf far_src;     // int32 source record positions of every proxy item, item by item
    DevBuf ranges_a;    // Range [n_ra]
    DevBuf ranges_b;    // Range [n_rb]
    DevBuf inst;        // Instance[ninst]
    int ninst = 1;
    bool batched = false;
    DevBuf charge_nodes; // int32 [n_charge] nodes whose proxies carry charges (BLTC)
    // upward pass (BLTC): items of <= FSS_UP_CHUNK records of one charge node;
    // nodes with several items sum their partial moments in a second pass
    int64_t n_up = 0, n_up_multi = 0, n_up_partial = 0, n_up_small = 0; // items <= 32 records first
    DevBuf up_items;    // int4 [n_up] {node, first record, records, partial index or -1}
    DevBuf up_multi;    // int4 [n_up_multi] {node, first partial, end partial, 0}
    DevBuf proxy_xyz;   // double4 [nn * p] static proxy positions (w unused)
    DevBuf src64;       // double4 [p0 + nn * p] source records (see above)
    DevBuf src32;       // float4 [p0 + nn * p], then float [nn * p] planar offsets
    DevBuf srcnode;     // int32 [p0 + nn * p] node of every source position (mixed precision)
    int64_t pairs_near = 0, pairs_far = 0;
};

// SAL state: series coefficients c_n (n = 0..nmax, c_0 = 0), the tabulated
// series on a uniform s-grid, and the learned kernel's parameters.
struct Sal {
    int nmax = 0;
    int64_t M = 0;       // table points
    double A = 0;        // coefficient of the analytic 1/(2s) - 1 part
    double g0 = 0;       // series at theta = 0 (self term)
    double mu = 0, sigma = 1; // normalisation of the learned remainder
    double s_min = 1e-3;      // the network input maps log s from [s_min, 1] onto [-1, 1]
    DevBuf c, tab, P, Pm, Pv, w;
    DevBuf mlpop; // the network in the form of its matrix-core evaluation (MlpOp, fss_sal_dev.h)
    bool has_mlp = false;
    int64_t adam_t = 0;
};

// Triangles of levels 0 .. levels-1 (levels concatenated): fixed by the depth, so
// they are computed once per context for its deepest tree.
struct Geo {
    int levels = 0;
    DevBuf xyz;  // 9 doubles per triangle (vertex coordinates, tree_tri_verts order)
    DevBuf info; // 4 doubles per triangle (centre, radius)
    // of the nodes, levels 0 .. levels-2
    DevBuf tinv; // 9 doubles: rows r_m with barycentric c_m = r_m . p
    DevBuf aux;  // double2: norm of the centre, arc radius of the cap
};

// Scratch of tree_build, kept between builds while it is small (BUILD_SCRATCH_KEEP).
struct BuildScratch {
    // info: BuildInfo, then the build's other arrays that start at zero (ZeroParts, fss_tree.hip)
    DevBuf info, cub, k0, k1, v0, v1, ek0, ek1, ev0, ev1, f0, f1, act, blk, per, pos, keys,
        keys2, vals, vals2, rcnt, rpos, rkeys, prox_one, cnt, off;
    std::vector<DevBuf *> all()
    {
        return {&info, &cub, &k0,  &k1,  &v0,   &v1,    &ek0,  &ek1,   &ev0,  &ev1,  &f0,    &f1,       &act, &blk,
                &per, &pos, &keys, &keys2, &vals, &vals2, &rcnt, &rpos, &rkeys, &prox_one, &cnt, &off};
    }
};

// Workspace of the remesh: missed targets, counters, and the triangle bins of
// the full search.
struct Remesh {
    DevBuf miss, cnt, tri, count, start, scan, place, cap, bin, odd;
};

// Page-locked host memory for the few words that a call reads back: a copy to
// pageable memory takes 23 us with its wait, one to page-locked memory 15.  Taking
// it costs 70 us, so contexts hand theirs on (words_take and ~HostWords in
// fss_api.cpp: at most 16 wait, the others are freed).
struct HostWords {
    static constexpr size_t BYTES = 4096;
    void *p = nullptr;
    HostWords() = default;
    HostWords(const HostWords &) = delete;
    HostWords &operator=(const HostWords &) = delete;
    ~HostWords();
};
// bytes from the device after everything before them on the context's stream;
// waits for them
fss_status read_back(fss_ctx *ctx, void *dst, const void *src, size_t bytes);

// Device time stamps of each velocity call in a ring of RING slots, kept without
// synchronizing; the mean over the slots since the last reset is read with
// fss_timing_mean().
struct Timing {
    static constexpr int RING = 256;
    // a slot: starts of the stage, the far kernel, the main kernel and what
    // follows it, then the ends of the stage's last blocks (see stamp_end)
    enum { START = 0, FAR = 1, MAIN = 2, MAIN_END = 3, END = 4, ENDS = 64, SLOT = END + ENDS };
    DevBuf stamps;      // uint64 [RING][SLOT], ticks of the device's constant clock
    double ms_per_tick = 0;
    uint8_t have[RING] = {}; // bits of the start stamps that the call's kernels write
    int64_t calls = 0;  // calls recorded since the last reset
    int cur = -1;       // slot of the current call
    bool valid = false;
    hipStream_t stream = nullptr; // of the last timed call
    bool streams = false; // the window's calls ran on more than one stream
    uint64_t *slot() const { return stamps.as<uint64_t>() + (int64_t)cur * SLOT; }
};

// begin a timed call: picks the next ring slot
inline void timing_begin(Timing &t, hipStream_t s)
{
    t.streams = t.calls > 0 && (t.streams || t.stream != s);
    t.stream = s;
    t.cur = (int)(t.calls % Timing::RING);
    t.calls++;
    t.have[t.cur] = 0;
}
// a stage's milliseconds: total, main kernel, far kernel (0 without one).  Waits for
// the context's stream, or for the device where calls ran on another.
fss_status timing_read(fss_ctx *ctx, int64_t first, int64_t count, double *stage, double *main, double *far);

// Time stamps by the kernels themselves (ts null: none).  The first block of a
// kernel starts it; at the end every block writes the clock to one of ENDS places,
// the last writer of each being the last to finish there, and the stage ends with
// the latest.  (HIP events around the kernels cost 4.5 us each on the stream:
// 22 of the 35 us of a direct sum of 2,562 particles.)
__device__ inline void stamp_start(uint64_t *ts, int which)
{
    if (ts && blockIdx.x == 0 && threadIdx.x == 0) ts[which] = wall_clock64();
}
__device__ inline void stamp_end(uint64_t *ts)
{
    if (ts && threadIdx.x == 0) ts[Timing::END + (blockIdx.x & (Timing::ENDS - 1))] = wall_clock64();
}

} // namespace fss

struct fss_ctx {
    fss_config cfg{};
    hipStream_t stream = nullptr;
    bool own_stream = false;
    bool batch_part = false; // tree_build of one batch instance: the merged plan is finished once
    fss::Interp interp;
    fss::Tree tree;
    fss::Timing timing;
    fss::Sal sal;
    fss::Remesh remesh;
    fss::Geo geo;
    fss::BuildScratch build;
    fss::HostWords words;

    // device constants
    fss::DevBuf d_lu, d_perm, d_vinv, d_pts;

    // per-stage workspace
    fss::DevBuf direct;  // partial sums or packed records of the direct sum
    fss::DevBuf out3;    // 3 doubles SoA [p0] per-position partial velocities
    fss::DevBuf phi;     // 3*p doubles per proxy work item (partial proxy values)
    fss::DevBuf alpha;   // 3*p doubles per interpolant slot
    fss::DevBuf upart;   // p doubles per partial moment of the upward pass
    fss::DevBuf acc3;    // 3 doubles per record: per-particle sums in tree order
    int near_r = 0;      // targets per lane of the near kernel: 2, 4 or 0 (4 in FP64, 2 in FP32)
    fss::DevBuf rk_k;    // 4 stages x 4 fields x n
    fss::DevBuf rk_y;    // stage state 4 x n
    fss::DevBuf rk_t;    // state and areas in tree order, 5 x n

    // hipGraph of one RK4 step
    hipGraph_t graph = nullptr;
    hipGraphExec_t graph_exec = nullptr;
    const void *graph_key[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    int64_t graph_n = 0;
    double graph_dt = 0;
    int graph_tree = -1;
    int graph_near_r = -1;
    uint64_t graph_epoch = 0; // alloc_epoch() when the graph was captured
    bool capturing = false; // inside hipStreamBeginCapture: no time stamps
};

namespace fss {

// ---- kernels / launchers (fss_tree.hip) ----
fss_status tree_build(fss_ctx *ctx, const double *x, const double *y, const double *z, int64_t n);
// source lists, item order and upward-pass items of single and batched plans;
// called last by both builders, and waits for the stream
fss_status plan_finish(fss_ctx *ctx);
void build_scratch_trim(BuildScratch &b);
fss_status tree_export(fss_ctx *ctx, int32_t *loc, uint8_t *found, int32_t *counts,
                       int32_t *offsets, int32_t *ids, int32_t *inter, double *tri_info,
                       double *tri_xyz);

// ---- interpolation constants (fss_api.cpp) ----
fss_status interp_setup(fss_ctx *ctx);

// ---- RK4 update at the end of an evaluation (fss_rk4_dev.h) ----
struct RkNext {
    enum { NONE = 0, STAGE = 1, STEP = 2 };
    int mode = NONE;
    double *x, *y, *z, *vort; // state of the step; STEP writes the new one here
    const double *k;          // STEP: velocities of the first three stages, 4 n each
    double *ys;               // STAGE: the next stage's state, 4 n
    int64_t n;
    double fac, omega;
};
// the update as a kernel of its own, from stored velocities (fss_rk4.hip)
fss_status rk4_next(fss_ctx *ctx, const RkNext &r, const fss_velocity &k);

// ---- evaluation (fss_eval.hip) ----
// tree_order: the arrays are in tree order (element i belongs to main record i;
// only for a tree without exception records).  next: an RK4 update to take with
// the velocities; its state may be the evaluated one.  STEP leaves out unwritten.
fss_status velocity_tree(fss_ctx *ctx, const fss_particles *p, fss_velocity *out, bool tree_order = false,
                         const RkNext &next = RkNext{});
// source records of a new plan (room for the particles', the proxies' laid down)
fss_status proxy_records(fss_ctx *ctx);

// ---- direct sum (fss_direct.hip) ----
fss_status velocity_direct(fss_ctx *ctx, const fss_particles *p, const int64_t *idx, int64_t m,
                           fss_velocity *out, bool force_fp64, const RkNext &next = RkNext{});

// allocation-free direct sum (fss_direct.hip): workspace in a file-scope device
// array per GPU (FSS_DIRECT_SCRATCH_BYTES of records and more), whose address
// direct_scratch_setup resolves once per device (that device current)
fss_status direct_scratch_setup(int device);
fss_status velocity_direct_noalloc(fss_ctx *ctx, const fss_particles *p, fss_velocity *out);

// ---- RK4 (fss_rk4.hip) ----
fss_status rk4_step(fss_ctx *ctx, double *x, double *y, double *z, double *vort,
                    const double *area, int64_t n, double dt, int use_tree);
fss_status rk4_run_graph(fss_ctx *ctx, double *x, double *y, double *z, double *vort,
                         const double *area, int64_t n, double dt, int use_tree, int steps);
fss_status project_points(fss_ctx *ctx, double *x, double *y, double *z, double *vort, int64_t n);

// FP64 records + BLTC charges of the current tree for a stage (fss_eval.hip)
fss_status tree_sources64(fss_ctx *ctx, const fss_particles *pp, uint64_t *ts);
// SAL convolution by the treecode (fss_sal_tree.hip)
fss_status sal_tree(fss_ctx *ctx, const fss_particles *pp, int kind, double *out);

// ---- remesh (fss_remesh.hip) ----
fss_status remesh(fss_ctx *ctx, const double *ax, const double *ay, const double *az, const double *avort,
                  const double *atr, const int32_t *tris, int64_t ntri, const int32_t *vt_off,
                  const int32_t *vt_idx, const double *x, const double *y, const double *z, double *vort,
                  double *tr, int32_t *tri_out, int64_t n, double omega, int64_t *n_fallback, int64_t *n_missing);

// ---- leaf-size autotuner (fss_tune.cpp) ----
int levels_for(int64_t n, double occupancy);
fss_status autotune_levels(fss_ctx *ctx, const fss_particles *pp, int lmin, int lmax, int reps, int *best,
                           double *ms);
fss_status autotune(fss_ctx *ctx, const fss_particles *pp, const fss_tune_point *cand, int ncand,
                    const int64_t *idx, int64_t m, double max_rel_l2, int reps, int *best, double *ms,
                    double *err);

// ---- batched instances (fss_batch.cpp) ----
fss_status batch_build(fss_ctx *ctx, int ninst, const int64_t *ns, const int *levels, const double *x,
                       const double *y, const double *z);

// ---- SAL (fss_sal.hip) ----
fss_status sal_set_series(fss_ctx *ctx, const double *c_host, int nmax, int64_t table_points, double A);
fss_status sal_series_eval(fss_ctx *ctx, const double *s_dev, int64_t m, double *g_dev);
fss_status sal_kernel_eval(fss_ctx *ctx, int kind, const double *s_dev, int64_t m, double *g_dev);
fss_status sal_mlp_params(fss_ctx *ctx, float *host, int set);
fss_status sal_mlp_init(fss_ctx *ctx, uint64_t seed);
fss_status sal_mlp_train(fss_ctx *ctx, int steps, int64_t nsamp, double lr, double s_min,
                         uint64_t seed, double *final_loss);
// matrix-core operand table of the current network parameters
fss_status sal_mlp_prepare(fss_ctx *ctx);
fss_status sal_mlp_grad(fss_ctx *ctx, const float *x_host, const float *y_host, int64_t m,
                        float *grad_host, float *loss_host);
fss_status sal_direct(fss_ctx *ctx, const double *x, const double *y, const double *z,
                      const double *eta, const double *area, int64_t n, const int64_t *idx,
                      int64_t m, int kind, double *out);
int sal_nparam();

inline int64_t div_up(int64_t a, int64_t b) { return (a + b - 1) / b; }

} // namespace fss
