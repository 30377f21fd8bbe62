/*
 * FP64 walk from interaction lists (plain form, precision NBHIP_PRECISION_FP64)
 * on gfx950, for states too small to fill the chip with one lane per body.
 *
 * The streaming walk (walk.hip) is a serial chain per wavefront of 64 bodies:
 * a scalar load, the test, the wave's vote, the branch, and an interaction
 * whose square root and quotients depend on each other, some 1200 cycles a
 * node step and 2000-3500 steps.  20 000 bodies are 313 such wavefronts on
 * 1024 SIMDs: 1.5 ms, of which the arithmetic fills a tenth.  Here the chain
 * is cut in two:
 *
 *  1. k_list_build, a workgroup per 64 consecutive sorted bodies, finds every
 *     node that any of them can meet, breadth first (all nodes of a level at
 *     once): a node is decided by the bodies' bounding box where its nearest
 *     point already passes the test (every body accepts) or its farthest point
 *     fails it (every body opens), and by the 64 tests themselves otherwise.
 *     Nodes that some body accepts are the list; it is put into pre-order
 *     (subtree sizes up the levels, places down them).
 *  2. k_walk_list, a wavefront per 8 (or 4) bodies, goes through the list in
 *     order: 64 entries at a time are tested against its own bodies, those
 *     that none of them accepts or that lie inside one accepted by all are
 *     dropped, and the others are taken 8 (16) at a time: lane (b, s) tests
 *     and evaluates entry s for body b.
 *
 * The reference's walk (nbGravity, nbody/src/nbody_grav.c:42-124) is kept to
 * the bit: the box only replaces decisions that are the same for every body
 * (rounding is monotone, so a box's nearest and farthest point bound the
 * computed squared distances of the bodies in it), a body's own test decides
 * the rest, a body skips what lies inside a node it has accepted (its place
 * in the walk, lp, as in the streaming walk), and its terms are added in
 * pre-order: the lanes leave their nine terms in LDS and one lane per (body,
 * component) adds them entry by entry, the reference's three additions each;
 * a lane that does not interact leaves zeros, which change no bit of the sum.
 *
 * Where a group's nodes do not fit its list (NBH_LIST_CAP) the whole state is
 * left to the streaming walk, which runs after this one.
 *
 * Measured (lists + walk against the streaming walk, BH86 theta = 0.5 with
 * quadrupoles): 1000 bodies 120 : 386 us, 4000 202 : 890, 20 000 413 : 1520,
 * 50 000 968 : 1795, 100 000 1868 : 2445; 200 000, with a batch fetched ahead,
 * 4200 : 3460 -- so up to
 * NBH_LIST_BODIES (131 072).  At 20 000 bodies the walk is 335 us (its
 * vector instructions alone 170) and the lists 79.  Beyond, each SIMD has
 * enough streaming waves to hide their chain, and the lists' LDS traffic
 * (17 LDS instructions per batch) no longer pays.
 */
#include "nbhip_list.h"
#include "nbhip_walk.h"

#include <type_traits>

#define NBH_LIST_KEEP (1u << 31)      /* build entry: goes into the list */
#define NBH_LIST_OPEN (1u << 30)      /* its children are entries too */
#define NBH_LIST_Q ((1u << 27) - 1u)  /* pre-order index; bits 27..29: children - 1 */

/* Squared distances from a node to the nearest and the farthest point of a
 * box, in the walk's operation order. */
struct ListBox {
    double lox, loy, loz, hix, hiy, hiz;
    __device__ __forceinline__ void dist(double x, double y, double z, double& near2,
                                         double& far2) const
    {
        const double ax = lox - x, bx = x - hix, ay = loy - y, by = y - hiy, az = loz - z,
                     bz = z - hiz;
        const double nx = fmax(fmax(ax, bx), 0.0), ny = fmax(fmax(ay, by), 0.0),
                     nz = fmax(fmax(az, bz), 0.0);
        const double fx = fmax(fabs(ax), fabs(bx)), fy = fmax(fabs(ay), fabs(by)),
                     fz = fmax(fabs(az), fabs(bz));
        near2 = nz * nz + (ny * ny + nx * nx);
        far2 = fz * fz + (fy * fy + fx * fx);
    }
};

__device__ __forceinline__ double nbh_wmin(double v)
{
    for (int off = 32; off > 0; off >>= 1) v = fmin(v, __shfl_xor(v, off, 64));
    return v;
}

/* The box of the wave's valid bodies. */
__device__ __forceinline__ ListBox nbh_list_box(bool valid, const double4& p)
{
    ListBox b;
    b.lox = nbh_wmin(valid ? p.x : INFINITY);
    b.loy = nbh_wmin(valid ? p.y : INFINITY);
    b.loz = nbh_wmin(valid ? p.z : INFINITY);
    b.hix = nbh_wave_max(valid ? p.x : -INFINITY);
    b.hiy = nbh_wave_max(valid ? p.y : -INFINITY);
    b.hiz = nbh_wave_max(valid ? p.z : -INFINITY);
    return b;
}

/* Interaction list of each 64-body group: list[g * NBH_LIST_CAP ..), length
 * llen[g]; scal->list_over where one does not fit.  All waves hold the group's bodies
 * (lane = body) for the box and share the nodes of a level. */
#define NBH_LB 512                    /* threads of k_list_build */
__global__ __launch_bounds__(NBH_LB) void k_list_build(const NodeW* __restrict__ node,
                                                    const double4* __restrict__ spos,
                                                    const int* __restrict__ simid_s,
                                                    const SimTab* __restrict__ sims,
                                                    const unsigned* __restrict__ nkid,
                                                    const unsigned* __restrict__ kbase,
                                                    const int* __restrict__ kid,
                                                    int* __restrict__ list,
                                                    int* __restrict__ llen,
                                                    DevScalars* __restrict__ scal, int n,
                                                    int multi)
{
    __shared__ unsigned s_q[NBH_LIST_CAP];            /* entry: flags and pre-order index */
    __shared__ unsigned short s_c[NBH_LIST_CAP];      /* first child's entry */
    __shared__ unsigned short s_n[NBH_LIST_CAP];      /* list entries in the subtree, then place */
    __shared__ int s_lev[65];                         /* first entry of each level */
    __shared__ double4 s_body[64];
    __shared__ int s_cnt, s_over, s_mix;
    if ((scal->status & (NBHIP_CELL_OVERFLOW_ERROR | NBHIP_ERROR)) || scal->halt) return;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int g = blockIdx.x;
    const int s = g * 64 + lane;
    const bool valid = s < n;
    const double4 p = valid ? spos[s] : make_double4(0.0, 0.0, 0.0, 0.0);
    const ListBox box = nbh_list_box(valid, p);
    const int sim = valid ? simid_s[s] : -1;
    if (tid < 64) s_body[tid] = p;
    if (tid == 0) {
        s_cnt = 0;
        s_over = (int) scal->list_over;               /* set meanwhile or not: one look for all */
    }
    __syncthreads();
    if (s_over) return;                               /* another group's did not fit */
    /* the roots of the group's simulations, in pre-order */
    if (!multi) {
        if (tid == 0 && sims[0].root >= 0) {
            s_q[0] = (unsigned) sims[0].root;
            s_cnt = 1;
        }
    } else if (tid < 64) {
        const int root = valid ? sims[sim].root : -1;
        bool first = root >= 0;
        for (int k = 1; k < 64; ++k) {
            const int o = __shfl(root, lane >= k ? lane - k : 0, 64);
            if (lane >= k && o == root) first = false;
        }
        const unsigned long long fm = __builtin_amdgcn_ballot_w64(first);
        int at = 0;
        for (unsigned long long r = fm; r; r &= r - 1)
            at += __builtin_amdgcn_readlane(root, __builtin_ctzll(r)) < root;
        if (first) s_q[at] = (unsigned) root;
        if (lane == 0) s_cnt = __popcll(fm);
    }
    __syncthreads();
    int lo = 0, hi = s_cnt, depth = 0;
    const int nroot = hi;
    const int nb = min(64, n - g * 64);
    /* entry i decided: kept or not, and its children's entries (all eight
     * loads of the child list in flight at once) */
    auto decide = [&](int i, unsigned q, bool open, bool keep, unsigned mask, unsigned kb) {
        unsigned e = q | (keep ? NBH_LIST_KEEP : 0u);
        if (open) {
            const int nk = __popc(mask);
            const int at = atomicAdd(&s_cnt, nk);
            if (at + nk > NBH_LIST_CAP || nk < 1 || nk > 8) {
                s_over = 1;
            } else {
                e |= NBH_LIST_OPEN | (unsigned) (nk - 1) << 27;
                s_c[i] = (unsigned short) at;
                int ch[8];
                #pragma unroll
                for (int j = 0; j < 8; ++j) ch[j] = kid[kb + min(j, nk - 1)];
                #pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (j < nk) s_q[at + j] = (unsigned) ch[j];
            }
        }
        s_q[i] = e;
    };
    while (lo < hi && depth < 64) {
        if (tid == 0) {
            s_lev[depth] = lo;
            s_mix = 0;
        }
        __syncthreads();
        /* what the group's box decides for every body; the rest to the work
         * list (s_n is free until the subtrees are counted) */
        for (int i = lo + tid; i < hi; i += NBH_LB) {
            const unsigned q = s_q[i];
            const NodeW w = node[q];
            const unsigned mask = nkid[q], kb = kbase[q];
            double near2, far2;
            box.dist(w.x, w.y, w.z, near2, far2);
            const bool cell = w.body < 0;
            if (!cell || near2 >= w.rcrit2) decide(i, q, false, true, mask, kb);
            else if (far2 < w.rcrit2) decide(i, q, true, false, mask, kb);
            else s_n[atomicAdd(&s_mix, 1)] = (unsigned short) i;
        }
        __syncthreads();
        /* the bodies' own tests, four lanes a node */
        const int nmix = s_mix;
        for (int t = tid; t < 4 * nmix; t += NBH_LB) {
            const int i = s_n[t >> 2];
            const unsigned q = s_q[i];
            const NodeW w = node[q];
            const unsigned mask = nkid[q], kb = kbase[q];
            int seen = 0;                             /* 1: a body accepts, 2: a body opens */
            #pragma unroll 4
            for (int k = t & 3; k < nb; k += 4) {
                const double4 c = s_body[k];
                const double dx = w.x - c.x, dy = w.y - c.y, dz = w.z - c.z;
                seen |= dz * dz + (dy * dy + dx * dx) >= w.rcrit2 ? 1 : 2;
            }
            seen |= __builtin_amdgcn_mov_dpp(seen, 0xB1, 0xF, 0xF, true);
            seen |= __builtin_amdgcn_mov_dpp(seen, 0x4E, 0xF, 0xF, true);
            if ((t & 3) == 0) decide(i, q, (seen & 2) != 0, (seen & 1) != 0, mask, kb);
        }
        __syncthreads();
        if (s_over) {
            if (tid == 0) scal->list_over = 1u;
            return;
        }
        lo = hi;
        hi = s_cnt;
        ++depth;
        __syncthreads();
    }
    if (lo < hi) {                    /* deeper than 63 levels: not a tree of ours */
        if (tid == 0) scal->list_over = 1u;
        return;
    }
    if (tid == 0) s_lev[depth] = hi;
    __syncthreads();
    /* list entries of each subtree, deepest level first */
    for (int l = depth - 1; l >= 0; --l) {
        for (int i = s_lev[l] + tid; i < s_lev[l + 1]; i += NBH_LB) {
            const unsigned e = s_q[i];
            int c = (e & NBH_LIST_KEEP) ? 1 : 0;
            if (e & NBH_LIST_OPEN) {
                const int a = s_c[i], nk = (int) ((e >> 27) & 7u) + 1;
                for (int j = 0; j < nk; ++j) c += s_n[a + j];
            }
            s_n[i] = (unsigned short) c;
        }
        __syncthreads();
    }
    /* places, from the roots down; a kept entry writes itself */
    int* out = list + (size_t) g * NBH_LIST_CAP;
    if (tid == 0) {
        int at = 0;
        for (int r = 0; r < nroot; ++r) {
            const int c = s_n[r];
            s_n[r] = (unsigned short) at;
            at += c;
        }
        llen[g] = at;
    }
    __syncthreads();
    for (int l = 0; l < depth; ++l) {
        for (int i = s_lev[l] + tid; i < s_lev[l + 1]; i += NBH_LB) {
            const unsigned e = s_q[i];
            int at = s_n[i];
            if (e & NBH_LIST_KEEP) out[at++] = (int) (e & NBH_LIST_Q);
            if (e & NBH_LIST_OPEN) {
                const int a = s_c[i], nk = (int) ((e >> 27) & 7u) + 1;
                for (int j = 0; j < nk; ++j) {
                    const int c = s_n[a + j];
                    s_n[a + j] = (unsigned short) at;
                    at += c;
                }
            }
        }
        __syncthreads();
    }
}

/* The terms in LDS: [component][term][lane], a write being one run of 64
 * doubles; the second half of the lanes two doubles on and rows of 76, which
 * keeps the adders' 16-byte reads (a body's slots, three components) on
 * different banks. */
#define NBH_TERM_ROW 76
__device__ __forceinline__ int nbh_term_at(int c, int t, int T, int lane)
{
    return (c * T + t) * NBH_TERM_ROW + lane + (lane >= 32 ? 2 : 0);
}

#define NBH_LW 2                      /* wavefronts per workgroup of k_walk_list */
template <int S, bool QUAD, bool AHEAD>
__global__ __launch_bounds__(64 * NBH_LW) void k_walk_list(const NodeW* __restrict__ node,
                                                           const double* __restrict__ nquad,
                                                           const double4* __restrict__ spos,
                                                           const unsigned* __restrict__ perm,
                                                           const int* __restrict__ simid_s,
                                                           SimTab* __restrict__ sims,
                                                           const int* __restrict__ list,
                                                           const int* __restrict__ llen,
                                                           double* __restrict__ oax,
                                                           double* __restrict__ oay,
                                                           double* __restrict__ oaz,
                                                           double* __restrict__ vx,
                                                           double* __restrict__ vy,
                                                           double* __restrict__ vz,
                                                           DevScalars* __restrict__ scal,
                                                           WalkOut o)
{
    constexpr int B = 64 / S;
    constexpr int T = QUAD ? 3 : 1;                   /* additions per component and entry */
    __shared__ int2 s_ring[NBH_LW][NBH_LIST_RING];
    __shared__ int s_next[NBH_LW][NBH_LIST_RING];
    __shared__ __align__(16) double s_term[NBH_LW][3 * T * NBH_TERM_ROW];
    /* list_over: the streaming walk's */
    if ((scal->status & (NBHIP_CELL_OVERFLOW_ERROR | NBHIP_ERROR)) | (unsigned) scal->halt |
        scal->list_over)
        return;
    const int w = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int first = (blockIdx.x * NBH_LW + w) * B;  /* the wave's first body */
    if (first >= o.n) return;
    const int g = first >> 6;
    const int len = llen[g];
    double* term = s_term[w];
    ListWave<S> L;
    L.start(node, nquad, s_ring[w], s_next[w], first, o.n, o.multi, o.all_eps2_pos != 0, spos,
            simid_s, sims, scal->nmassive);
    double acc = 0.0;                                 /* of body lane % B, component lane / B */

    L.template run<QUAD, AHEAD>(list + (size_t) g * NBH_LIST_CAP, len, [&](const ListRec& r, int cnt) {
        const ListHit h = L.hit(r, cnt);
        /* unused lanes: mass 0 and no quadrupole, at a harmless distance */
        const double m = h.use ? r.zm.y : 0.0;
        double t[9];
        auto eval = [&](auto P) {
            constexpr bool PL = decltype(P)::value;
            NbhRoot c;
            const double mor3 = nbh_mor3<PL>(m, h.r2, c);
            t[0] = mor3 * h.dx;
            t[1] = mor3 * h.dy;
            t[2] = mor3 * h.dz;
            if (QUAD) {
                const double qx = r.q0.x * h.dx + r.q0.y * h.dy + r.q1.x * h.dz;
                const double qy = r.q0.y * h.dx + r.q1.y * h.dy + r.q2.x * h.dz;
                const double qz = r.q1.x * h.dx + r.q2.x * h.dy + r.q2.y * h.dz;
                const double dQd = qx * h.dx + qy * h.dy + qz * h.dz;
                double d5 = nbh_dr5<PL>(h.r2, c);
                d5 = h.use ? d5 : 0.0;
                const double phiQ = nbh_phiq<PL>(d5, dQd, h.r2, c);
                t[3] = phiQ * h.dx;
                t[4] = phiQ * h.dy;
                t[5] = phiQ * h.dz;
                t[6] = -d5 * qx;
                t[7] = -d5 * qy;
                t[8] = -d5 * qz;
            }
            /* A body's quadrupole record is zero, an unused lane's mass and d5
             * too, and in the plain range everything they multiply is finite.
             * Outside it 1 / r^5 of a close body (itself: r^2 = eps2), the
             * quadrupole of a cell that this lane opens or the place of another
             * simulation's node may not be. */
            if (!PL) {
                #pragma unroll
                for (int k = 0; k < 3 * T; ++k)
                    t[k] = h.use & (k < 3 || h.nbody < 0) ? t[k] : 0.0;
            }
        };
        if (L.plain) eval(std::true_type()); else eval(std::false_type());
        #pragma unroll
        for (int c = 0; c < 3; ++c) {
            #pragma unroll
            for (int k = 0; k < T; ++k) term[nbh_term_at(c, k, T, lane)] = t[c + 3 * k];
        }
        nbh_wave_sync();
        if (lane < 3 * B) {
            const int c = lane / B;                   /* lane = c * B + body */
            double v[T][S];
            #pragma unroll
            for (int k = 0; k < T; ++k) {
                const double2* from = reinterpret_cast<const double2*>(
                    term + nbh_term_at(c, k, T, (lane % B) * S));
                #pragma unroll
                for (int u = 0; u < S / 2; ++u) {
                    const double2 x = from[u];
                    v[k][2 * u] = x.x;
                    v[k][2 * u + 1] = x.y;
                }
            }
            #pragma unroll
            for (int u = 0; u < S; ++u) {
                #pragma unroll
                for (int k = 0; k < T; ++k) acc += v[k][u];
            }
        }
        nbh_wave_sync();
    });

    /* the body's three components to one lane, and whether any slot met it */
    const unsigned long long mm = __builtin_amdgcn_ballot_w64(L.met);
    if (lane < 3 * B) term[lane] = acc;
    nbh_wave_sync();
    const int fb = first + lane;
    if (lane >= B || fb >= o.n) return;
    const unsigned long long bits = (mm >> (lane * S)) & ((1ull << S) - 1ull);
    const int fsim = simid_s[fb];
    if (bits == 0ull) atomicOr(&sims[fsim].incest, 1u);
    const double4 fp = spos[fb];
    nbh_walk_finish(o, fp.x, fp.y, fp.z, term[lane], term[B + lane], term[2 * B + lane], perm[fb],
                    oax, oay, oaz, vx, vy, vz);
}

/* The groups' lists for the current tree and bodies. */
void nbh_list_build(nbhip_state* st)
{
    if (st->n <= 0) return;
    hipLaunchKernelGGL(k_list_build, dim3((st->n + 63) / 64), dim3(NBH_LB), 0, st->stream,
                       st->node, st->spos, st->simid_s, st->sims, st->nkid, st->kbase, st->kid,
                       st->wlist, st->wlen, st->scal, st->n, st->nsim > 1);
}

void nbh_walk_list(nbhip_state* st, const WalkOut& o, double* oax, double* oay, double* oaz)
{
    hipStream_t s = st->stream;
    const int n = st->n;
    if (n <= 0) return;
    nbh_list_build(st);
#define NBH_WL(S, Q, A)                                                                        \
    hipLaunchKernelGGL((k_walk_list<S, Q, A>), dim3((n + 64 * NBH_LW / S - 1) / (64 * NBH_LW / S)),    \
                       dim3(64 * NBH_LW), 0,                                                   \
                       s, st->node, st->nquad, st->spos, st->perm, st->simid_s, st->sims,      \
                       st->wlist, st->wlen, oax, oay, oaz, st->vx, st->vy, st->vz, st->scal, o)
    /* Four bodies a wavefront, sixteen entries a batch, while that leaves SIMDs
     * idle: 1000 bodies 120 against 151 us (lists and walk), 4000 202 against
     * 268, 20 000 473 against 413.
     * Eight: fetching a batch ahead takes 160 registers, three waves a SIMD;
     * with more waves than that makes room for (24 576 bodies), a fourth wave
     * hides more than the fetch: 20 000 bodies 338 against 352 us (the walk),
     * 40 000 684 against 650, 100 000 1878 against 1695. */
    if (n <= NBH_LIST_WIDE) {
        if (st->ctx.use_quad) NBH_WL(16, true, true); else NBH_WL(16, false, true);
    } else if (n <= NBH_LIST_AHEAD) {
        if (st->ctx.use_quad) NBH_WL(8, true, true); else NBH_WL(8, false, true);
    } else {
        if (st->ctx.use_quad) NBH_WL(8, true, false); else NBH_WL(8, false, false);
    }
#undef NBH_WL
}
