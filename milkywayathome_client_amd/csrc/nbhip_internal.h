/*
 * Internal declarations of the nbhip library (not part of the C ABI).
 *
 * HBM layout of one simulation (N bodies, node capacity C):
 *   bodies, original order, SoA FP64 : px py pz vx vy vz m ax ay az   (80 B/body)
 *   sort: 64-bit Morton word (levels 1-21) + 32-bit body index, ping-pong
 *   sorted bodies: spos (x y z m, 32 B) and 63-bit fixed-point coordinates
 *     su (3 x 8 B) of the massive bodies, used for the 189-bit Morton prefix
 *   adjacent prefixes dadj of the sorted massive bodies and their
 *     min-hierarchy (the binary radix tree, Karras 2012, is never stored:
 *     it is the Cartesian tree of dadj, found by nearest-smaller searches)
 *   node table in pre-order (the reference's More/Next threading order):
 *     NodeW (48 B: centre of mass, mass, rcrit2, Next index, body) + quad
 *     (48 B) + build-only level/parent/child counters/midpoint.
 */
#ifndef NBHIP_INTERNAL_H
#define NBHIP_INTERNAL_H

#include <hip/hip_runtime.h>
#include "../../include/nbhip.h"

/* Walk record of one node.  body >= 0: a massive body (its sorted index);
 * body < 0: a cell.  next: pre-order index of Next(node). */
struct __attribute__((aligned(16))) NodeW {
    double x, y, z, m;
    double rcrit2;
    int next;
    int body;
};

/* Walk record of the mixed-precision walk (64 B, one scalar load).
 * The position stays FP64: the walk forms each displacement as one FP64
 * subtraction rounded once to FP32, exact to FP32 however far the record and
 * the body are from the origin.  rcrit2 is -1 for bodies (always accepted);
 * q[6] is the quadrupole in FP32 (zero for bodies). */
struct __attribute__((aligned(16))) NodeF {
    double x, y, z;
    float m, rcrit2;
    int next, body;
    float q[6];
};

/* Record of the group walk's table, in which every cell's children occupy
 * one contiguous block (slots 0 .. nsim-1 hold the simulations' roots).
 * Position FP64 (displacements are formed relative to the group in FP64 and
 * rounded once); rcrit2 is the squared critical radius times the open scale,
 * rounded towards +infinity to FP32 (so the group test never accepts what
 * the FP64 criterion opens), -1 for bodies.  Cells: link = first child slot,
 * count = children (1..8); bodies: link = sorted body index, count = 0. */
struct __attribute__((aligned(16))) NodeG {
    double x, y, z;
    float m, rcrit2;
    int link, count;
    float q[6];
};

/* Exact criterion: the sources of a simulation of n bodies are summed in
 * this many consecutive segments (one per grid row), 1 below 4096 bodies --
 * there the sum is the reference's, bit for bit.  Enough of them that the
 * last round of workgroups is short: 20000 bodies are 79 x 32 workgroups, 9.9
 * a CU (9 segments: 2.8, three rounds for two and three quarters;
 * gradient of four steps 10.98 against 10.50 ms). */
__host__ __device__ inline int nbh_exact_segments(int n)
{
    const int s = n / 256;
    return n < 4096 ? 1 : (s > 32 ? 32 : s);
}

/* Per-simulation device record (one per dwarf of a batch; one for a single
 * simulation). */
struct SimTab {
    double rsize;                  /* st->tree.rsize, persists, grows only */
    double key_scale;              /* 2^63 / rsize */
    double eps2;
    unsigned long long xyzmax_bits;/* max |x_i| of the last bbox pass */
    int body_off, body_n;          /* bodies, original order */
    int first;                     /* first sorted massive body, -1 if none */
    int root, end;                 /* pre-order segment [root, end), -1 if none */
    int maxdepth;
    unsigned flags;                /* sticky NBHIP_* bits of this simulation */
    unsigned incest;               /* a body of this simulation missed itself */
    unsigned odd_mass;             /* a mass was nonzero and outside the range of the unscaled
                                      divisions (nbh_plain_range), or a position not finite, or
                                      none was looked at yet */
    unsigned odd_seen;             /* the same, gathered by the bbox pass that is running */
};

/* Device-resident scalars shared by all simulations of a state. */
struct DevScalars {
    int nmassive;                  /* massive bodies, all simulations */
    int ncell;
    int nnode;
    int maxdepth;
    unsigned status;               /* sticky global bits (overflow, internal error) */
    int sim_bits;                  /* key bits holding the simulation id */
    unsigned long long counters[5];/* body-body, body-cell, opened, wave node steps,
                                      group far-field (cell, group) pairs */
    unsigned list_over;            /* a group's interaction list of this tree did not fit: the
                                      whole state streams */
    int halt;                      /* a step ended with a fatal status: later steps do nothing */
    unsigned steps_done;           /* KDK steps completed on the device */
    int level_count[64];           /* cells per level */
    int level_fill[64];
    int level_off[65];             /* exclusive scan of level_count */
    unsigned group_mean;           /* group walk: mean predicted group cost of the last walk */
};

/* Walk tuning picked by the autotuner (nbhip_autotune). */
struct WalkTune {
    int block;                     /* threads per workgroup: 64, 128 or 256 */
    int batch;                     /* mixed walk: node block per FP32 partial sum (power of 2);
                                      group walk: LDS interaction-list depth (64, 128, 256) */
};

/* Group walk tasks: the sub-groups of a 64-body group predicted to cost
 * more than NBH_GW_SPLIT_COST times the mean group are shared out among up
 * to 8 waves (runs of whole sub-groups, each run at most that cost where a
 * sub-group allows); at most NBH_GW_EXTRA_TASKS such extra waves per walk. */
#define NBH_GW_EXTRA_TASKS 1024
#define NBH_GW_SPLIT_COST 2
__host__ __device__ inline int nbh_group_tasks(int n) { return (n + 63) / 64 + NBH_GW_EXTRA_TASKS; }

/* Min-hierarchy over the adjacent prefixes, in dadj's allocation after its
 * n entries: level 0 is dadj[0..M), level L >= 1 holds the minimum of each 16
 * entries of level L-1 (size ceil(M / 16^L)), every level starting on a
 * multiple of 16 entries, up to the first level of at most 16 entries. */
struct NbhDHier {
    int top;
    int size[9];
    int off[9];
};
__host__ __device__ inline NbhDHier nbh_dhier(int n, int M)
{
    NbhDHier h;
    h.top = 0;
    h.size[0] = M;
    h.off[0] = 0;
    int at = (n + 15) & ~15;
    while (h.size[h.top] > 16 && h.top < 8) {
        const int s = (h.size[h.top] + 15) / 16;
        ++h.top;
        h.size[h.top] = s;
        h.off[h.top] = at;
        at += (s + 15) & ~15;
    }
    return h;
}
/* dadj's allocation: n prefixes and the hierarchy's levels for M <= n */
__host__ __device__ inline size_t nbh_dadj_cap(int n)
{
    size_t at = ((size_t) n + 15) & ~(size_t) 15, s = (size_t) n;
    while (s > 16) {
        s = (s + 15) / 16;
        at += (s + 15) & ~(size_t) 15;
    }
    return at + 16;
}

/* Interaction lists of the FP64 list walk: entries per 64-body group (LDS of
 * the list's build: 8 bytes an entry). */
#define NBH_LIST_CAP 8192
/* states of at most this many bodies walk lists (walk_list.hip has both
 * sides' times), and of at most this many with sixteen entries a batch */
#define NBH_LIST_BODIES (1 << 17)
#define NBH_LIST_WIDE 8192
#define NBH_LIST_AHEAD 24576   /* and of at most this many a batch is fetched ahead */

/* Where the lists of a state do not fit, it streams, and what bounds that is
 * the wave with the longest chain of nodes.  Fewer bodies a wave meet fewer
 * nodes, and up to a wave a SIMD it costs nothing: 8, 16, 32 or 64 bodies, the
 * fewest that leave at most NBH_STREAM_WAVES waves.  A force at theta 0.2 with
 * 512, 1024 and 2048 of them, and from the streaming walk alone with 64 bodies
 * a wave, us: 9000 bodies 3019, 2948, 3114, 3618; 20000 5150, 4912, 5972,
 * 5934; 50000 8173, 8168, 10806, 9510. */
#define NBH_STREAM_WAVES 1024
inline int nbh_stream_bodies(int n)
{
    int per = 8;
    while (per < 64 && n > per * NBH_STREAM_WAVES) per *= 2;
    return per;
}

/* Mixed and coherent walks of at most NBH_PIECE_BODIES bodies are cut into
 * NBH_PIECES parts (8 and 16 parts, one wave, us per mixed walk: 2x10^4
 * bodies 312, 230, 836; 10^5 740, 689, 1196; 2x10^5 1230, 1136, 1573; 4x10^5
 * 2184, 2198, 2289; at 10^6 8 parts 5433, one wave 5154).  The 16 waves of
 * the same bodies in one workgroup instead: 2450 at 10^5 -- waves that walk
 * the same nodes have to share a scalar cache.  Consecutive workgroups on
 * consecutive XCDs instead of one stretch of bodies an XCD: 810. */
#define NBH_PIECES 16
#define NBH_PIECE_BODIES (1 << 18)
/* Bodies of at most NBH_PINNED_BODIES leave the device through the state's
 * page-locked block, written by the packing kernel itself: with the status
 * read the same way, an eager step of 1021 bodies and its read-back take 233
 * us against 450 with nine copies and waits and strided loops of the host.
 * More bodies are packed in device scratch and copied an array at a time
 * (4 steps of 10^6 bodies and the read-back 53.0 ms against 57). */
#define NBH_PINNED_BODIES 4096
#define NBH_SORT_TILE 2048   /* keys per radix-sort block: 256 threads x 8 */
#define NBH_SCAN_TILE 4096   /* items per scan block: 1024 threads x 4 */

/* Adjoint bookkeeping (FP64 states only): checkpoints of the forward run
 * every `every` steps, one recomputed segment, and the adjoint vectors.
 * A state slot holds 9 arrays of n doubles: x y z vx vy vz ax ay az. */
struct NbhAdjoint {
    unsigned nsteps, every, nckpt;
    double* ckpt;                 /* nckpt slots */
    SimTab* ckpt_tab;             /* nckpt * nsim */
    double* seg;                  /* every + 1 slots */
    SimTab* seg_tab;              /* (every + 1) * nsim */
    double* fin;                  /* final forward state, one slot */
    SimTab* fin_tab;
    double* g;                    /* gx gy gz | gvx gvy gvz | gax gay gaz | gm: 10 n */
    double* gdt;                  /* nsim */
    double* gnode;                /* 10 * node_cap: d/d(cm x y z, mass, quad[6]) */
    int ready;
};

struct nbhip_state {
    nbhip_ctx ctx;
    int device;
    int n;                        /* bodies, all simulations */
    int nsim;
    int sim_shift;                /* key bit where the simulation id starts */
    int top_levels;               /* Morton levels in the sort word */
    int node_cap;
    int sort_blocks;
    hipStream_t stream;

    double *px, *py, *pz, *vx, *vy, *vz, *m, *ax, *ay, *az;
    int *simid;                   /* simulation of each body, original order */

    unsigned long long *key, *key_alt;
    unsigned *perm, *perm_alt;
    unsigned *hist;
    unsigned *dtot;               /* per-digit totals of one radix pass */

    double4 *pos4;                /* x, y, z, m per body, original order (build input) */
    double4 *spos;
    int *simid_s;                 /* simulation of each sorted body */
    unsigned long long *su;       /* 3 per sorted body: ux, uy, uz */
    int *dadj;
    unsigned *cincl;              /* inclusive scan of cells-per-first-body */
    unsigned *scan_part;


    NodeW *node;
    double *nquad;                /* 6 per node */
    double *nmid;                 /* 3 per node (cells) */
    int *nnext;                   /* cells: pre-order index of Next(cell) (the walk record's
                                     next, kept compact for the summaries) */
    int *nlevel, *nparent, *nsim_node;
    int *level_list;              /* cell pre-order indices grouped by level */
    NodeF *nodef;                 /* mixed-precision walk records (precision MIXED) */
    NodeG *nodeg;                 /* group walk table (precision MIXED_GROUP): nsim + node_cap */
    unsigned *bcost;              /* group walk: per body (original order), its sub-group's work
                                     in the last walk */
    float *bbox;                  /* group walk: per body, its sub-group's box half-diagonal in
                                     the last walk */
    unsigned *gcost;              /* group walk: predicted work of each 64-body group, and
                                     its task count - 1 in bits 28..30 */
    uint2 *gtask;                 /* group walk: up to 8 tasks per group: (cost, lo | hi << 8) */
    int2 *gorder;                 /* group walk: [0].x = task count, then the tasks (group,
                                     lo | hi << 8) in dispatch order, costliest first */
    unsigned *nkid;               /* children per node */
    unsigned *kbase;              /* exclusive scan of nkid: each cell's child block */
    int *nrank;                   /* a node's rank among its parent's children (arrival order) */
    int *kid;                     /* child lists: kid[kbase[p] .. + nkid[p]) */
    int *blist;                   /* summaries: inside cells of each body block, by level */
    int *span, *span_sorted;      /* summaries: cells spanning body blocks / super-blocks */
    int *wlist, *wlen;            /* FP64 list walk: each 64-body group's nodes in pre-order
                                     (NBH_LIST_CAP slots) and their count */
    double *wsum;                 /* mixed walk in parts: each part's sums and their errors */
    unsigned *wmet;               /* and 0 where a body met its own record */
    double *exact_part;           /* Exact criterion: per-segment partial sums */
    int exact_seg;                /* Exact criterion: most segments of any simulation */

    DevScalars *scal;
    SimTab *sims;
    int *h_body_off, *h_body_n;   /* host copies */
    int all_eps2_pos;

    unsigned step;
    unsigned dev_steps;           /* DevScalars::steps_done at the last status read */
    double* best_buf;             /* bodies of the best-likelihood step: x y z vx vy vz */
    int best_kept;                /* best_buf holds the last run's best step */
    unsigned status;              /* host-side sticky status (all simulations) */
    unsigned *h_sim_status;       /* host-side sticky status per simulation */
    int have_tree;
    int profiling;
    hipEvent_t ev[6];
    float phase_ms[5];

    int h_level_count[64];        /* cells per level of the last eager build */
    int h_levels_valid;
    char *h_pinned;               /* page-locked: 64 level counts, scalars, SimTab rows, and the
                                     bodies of a state of at most NBH_PINNED_BODIES */
    struct DevScalars *h_scal;    /* within it */
    SimTab *h_sims;
    double *h_bodies;
    int *h_counts_pinned;         /* pinned landing buffer of the level-count readback */
    hipEvent_t ev_counts;         /* recorded after that readback */

    NbhAdjoint* adj;

    unsigned char* ignore;        /* per body, original order: left out of histograms */
    unsigned* hist_buf;           /* device counts + totals of nbhip_histogram */
    size_t hist_cap;              /* unsigned entries in hist_buf */
    double open_scale;            /* coherent walk: critical radius^2 factor (>= 1) */
    double group_far;             /* group walk: far-field expansion ratio (0: off) */
    char* disp_buf;               /* scratch of nbhip_histogram_dispersion (grow-only) */
    size_t disp_cap;              /* bytes in disp_buf */

    WalkTune tune;
    int use_graph;
    hipGraph_t graph;
    hipGraphExec_t graph_exec;
    int graph_ready;
};

/* launchers (tree.hip) */
void nbh_bbox(nbhip_state* st, int drift);
void nbh_build(nbhip_state* st, int graph_safe);
unsigned nbh_level_lists(nbhip_state* st);
void nbh_step_end(nbhip_state* st);
/* x, y, z of n bodies <-> n triples (asynchronous); raw copies of device
 * data by a kernel, which may write page-locked memory */
void nbh_pack3(hipStream_t s, int n, const double* x, const double* y, const double* z,
               double* out);
void nbh_unpack3(hipStream_t s, int n, const double* in, double* x, double* y, double* z);
void nbh_pack_bodies(nbhip_state* st, int off, int n, double* pos, double* vel, double* acc);
void nbh_export_status(nbhip_state* st);
/* the first `arrays` of x y z vx vy vz ax ay az and the SimTab rows <-> a slot */
void nbh_slot_copy(nbhip_state* st, double* slot, SimTab* tab, int arrays, int save);
void nbh_masses_changed(nbhip_state* st);
/* launchers (walk.hip) */
void nbh_walk(nbhip_state* st, int kick, int count, double* out_ax, double* out_ay,
              double* out_az, int self_only, const WalkTune* tune);
void nbh_list_build(nbhip_state* st);
void nbh_walk_list(nbhip_state* st, const struct WalkOut& o, double* out_ax, double* out_ay,
                   double* out_az);
void nbh_direct(nbhip_state* st, int nsample, const int* d_idx, double* d_acc);
/* launcher (walk_group.hip) */
struct WalkOut;
void nbh_walk_group(nbhip_state* st, const WalkOut& o, double* out_ax, double* out_ay,
                    double* out_az, const WalkTune& t, int count);
/* launcher (histogram.hip) */
void nbh_histogram(nbhip_state* st, const nbhip_histogram_params* hp, unsigned* d_counts,
                   unsigned* d_totals);
size_t nbh_disp_bytes(int cnt, size_t nbin);
const double* nbh_dispersion(nbhip_state* st, int off, int cnt, const nbhip_histogram_params* hp,
                             const nbhip_disp_params* dp, char* scratch_bytes);
/* scratch of the allocation-free entry point (histogram.hip) */
unsigned nbh_scratch_init(int device);
/* launchers (adjoint.hip) */
void nbh_adj_kick_end(nbhip_state* st, const double* a_next);
void nbh_adj_force(nbhip_state* st);
void nbh_exact_force(nbhip_state* st, int kick, double* oax, double* oay, double* oaz,
                     int use_pot);
void nbh_exact_adjoint(nbhip_state* st, double* g);
void nbh_adj_body(nbhip_state* st, int drift_kick, const double* v_prev, const double* a_prev);

#define NBH_CHECK(x)                                                         \
    do {                                                                     \
        hipError_t e_ = (x);                                                 \
        if (e_ != hipSuccess) {                                              \
            nbh_set_error("%s:%d: %s: %s", __FILE__, __LINE__, #x,           \
                          hipGetErrorString(e_));                            \
            return NBHIP_GPU_ERROR;                                          \
        }                                                                    \
    } while (0)

void nbh_set_error(const char* fmt, ...);

#endif
