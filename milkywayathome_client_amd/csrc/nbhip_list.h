/*
 * A wavefront's pass through its group's interaction list (walk_list.hip has
 * the method): the filter of 64 entries at a time against the wave's own
 * bodies, the batches of S entries, and each lane's decision.  Shared by the
 * list walk and its adjoint.
 */
#ifndef NBHIP_LIST_H
#define NBHIP_LIST_H

#include "nbhip_device.h"

/* Maximum over the S = 4, 8 or 16 consecutive lanes of a body. */
template <int S>
__device__ __forceinline__ int nbh_slots_max(int v)
{
    v = max(v, __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true));              /* xor 1 */
    v = max(v, __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true));              /* xor 2 */
    if (S >= 8) v = max(v, __builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true)); /* half row mirrored */
    if (S >= 16) v = max(v, __builtin_amdgcn_mov_dpp(v, 0x140, 0xF, 0xF, true)); /* row mirrored */
    return v;
}

/* v of one lane, uniform. */
__device__ __forceinline__ double nbh_lane_d(double v, int lane)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int) (unsigned) (b & 0xffffffffll), lane);
    const int hi = __builtin_amdgcn_readlane((int) (b >> 32), lane);
    return __longlong_as_double(((long long) hi << 32) | (unsigned) lo);
}

#define NBH_LIST_RING 128

/* A batch lane's node: record and quadrupole as loaded; cont has bit S - d
 * set where the entry d places back contains this one. */
struct ListRec {
    unsigned q, cont;
    double2 xy, zm, rl, q0, q1, q2;
};

/* Maximum over this lane and the lanes below it. */
__device__ __forceinline__ int nbh_scan_max(int v)
{
    /* row_shr 1, 2, 4, 8, then each row's last lane to the rows above
     * (lanes without a source read 0: the values are indices >= 0) */
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true));
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false)); /* row_bcast 15 */
    v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false)); /* row_bcast 31 */
    return v;
}

/* What a lane makes of its entry: the displacement, and whether its body
 * interacts with the node (r2 is then the softened squared distance, 1
 * otherwise). */
struct ListHit {
    double dx, dy, dz, r2;
    int nbody;                       /* the node's body, -1 for a cell */
    bool use;
};

/* lane = b * S + s: body b of the wave's B = 64 / S, slot s of the batch. */
template <int S>
struct ListWave {
    static constexpr int B = 64 / S;
    const NodeW* node;
    const double* nquad;
    int2* ring;                      /* LDS, NBH_LIST_RING each */
    int* rnext;
    int lane, b, slot, body;
    bool valid, plain, eps2_pos, met;
    double4 p;
    double eps2;
    int spare;                       /* an entry of the list: the node of lanes without one */
    int lp, end, self;               /* place in the body's walk, its simulation's end */
    double bx[B], by[B], bz[B];      /* the wave's bodies, uniform (past the last: the first) */

    __device__ __forceinline__ void start(const NodeW* node_, const double* nquad_, int2* ring_,
                                          int* rnext_, int first, int n, int multi,
                                          bool eps2_pos_, const double4* spos,
                                          const int* simid_s, const SimTab* sims, int nmassive)
    {
        node = node_;
        nquad = nquad_;
        ring = ring_;
        rnext = rnext_;
        lane = threadIdx.x & 63;
        b = lane / S;
        slot = lane % S;
        body = first + b;
        valid = body < n;
        const double4 f = spos[first];
        p = valid ? spos[body] : f;
        #pragma unroll
        for (int k = 0; k < B; ++k) {
            bx[k] = nbh_lane_d(p.x, k * S);
            by[k] = nbh_lane_d(p.y, k * S);
            bz[k] = nbh_lane_d(p.z, k * S);
        }
        const SimTab& st = sims[simid_s[valid ? body : first]];
        eps2 = st.eps2;
        lp = valid && st.root >= 0 ? st.root : INT_MAX;
        end = multi ? st.end : INT_MAX;
        self = valid && body < nmassive ? body : -2;
        eps2_pos = eps2_pos_;
        /* plain: every simulation of the group, whose nodes are in the list */
        bool odd = !nbh_plain_range(st);
        if (multi) {
            const int o = (first & ~63) + lane;
            odd = !nbh_plain_range(sims[simid_s[o < n ? o : first]]);
        }
        plain = __builtin_amdgcn_ballot_w64(odd) == 0ull;
        met = false;
        rnext[lane] = rnext[lane + 64] = 0;
        ring[lane] = ring[lane + 64] = make_int2(0, 0);
    }

    /* entries head .. head + S - 1 of the ring, cnt of them live */
    template <bool QUAD>
    __device__ __forceinline__ ListRec fetch(int head, int cnt) const
    {
        ListRec r;
        const int2 e = ring[(head + slot) & (NBH_LIST_RING - 1)];
        r.q = (unsigned) (slot < cnt ? e.x : spare);
        r.cont = (unsigned) e.y;
        /* 32-bit offsets: a body is the first of at most 64 cells, one a level */
        static_assert(65ull * NBH_LIST_BODIES * 48 < 1ull << 32, "node offsets");
        const unsigned off = r.q * 48u;
        const double2* rec =
            reinterpret_cast<const double2*>(reinterpret_cast<const char*>(node) + off);
        r.xy = rec[0];
        r.zm = rec[1];
        r.rl = rec[2];
        if (QUAD) {
            const double2* qr =
                reinterpret_cast<const double2*>(reinterpret_cast<const char*>(nquad) + off);
            r.q0 = qr[0];
            r.q1 = qr[1];
            r.q2 = qr[2];
        }
        return r;
    }

    __device__ __forceinline__ ListHit hit(const ListRec& r, int cnt)
    {
        ListHit h;
        const bool live = slot < cnt;
        const int q = (int) r.q;
        const long long link = __double_as_longlong(r.rl.y);
        const int next = (int) (unsigned) (link & 0xffffffffll);
        h.nbody = (int) (link >> 32);
        h.dx = r.xy.x - p.x;
        h.dy = r.xy.y - p.y;
        h.dz = r.zm.x - p.z;
        const double drSq = h.dz * h.dz + (h.dy * h.dy + h.dx * h.dx);
        /* a node passes by itself; it is met unless it lies inside one that
         * was accepted: before this batch (lp) or in it (cont) */
        /* A body's rcrit2 is 0, and it is accepted also where the distance is
         * no number.  (A cell of such a distance is opened; it is in the list
         * only for a body that is no number itself, and whose sum is none
         * either way.) */
        const bool pass = live & !(drSq < r.rl.x);
        const unsigned long long pm = __builtin_amdgcn_ballot_w64(pass);
        const unsigned mine = (unsigned) (pm >> (b * S)) << (S - slot);
        const bool here = pass & (q >= lp) & (q < end) & ((mine & r.cont) == 0u);
        lp = max(lp, nbh_slots_max<S>(pass ? next : 0));
        met |= here & (h.nbody == self);
        h.use = here & (eps2_pos | (h.nbody != self));
        h.r2 = h.use ? drSq + eps2 : 1.0;
        return h;
    }

    /* Every entry of the list, in order: batch(record, live entries).  AHEAD:
     * a batch's records are fetched while the one before is evaluated. */
    template <bool QUAD, bool AHEAD, class Batch>
    __device__ __forceinline__ void run(const int* lst, int len, Batch&& batch)
    {
        int head = 0, tail = 0, skip = 0;             /* skip: nothing before it is met by anyone */
        /* the filter's nodes one chunk ahead, their indices two */
        int q_next = lane < len ? lst[lane] : 0;
        NodeW nd_next = node[q_next];
        int q_after = 64 + lane < len ? lst[64 + lane] : 0;
        spare = __builtin_amdgcn_readfirstlane(q_next);
        nbh_wave_sync();
        for (int i0 = 0; i0 < len; i0 += 64) {
            const bool in = i0 + lane < len;
            const int q = q_next;
            const NodeW nd = nd_next;
            q_next = q_after;
            if (i0 + 64 < len) nd_next = node[q_next];
            q_after = i0 + 128 + lane < len ? lst[i0 + 128 + lane] : 0;
            int opens = 0;                            /* bodies that open this node */
            #pragma unroll
            for (int k = 0; k < B; ++k) {
                const double dx = nd.x - bx[k], dy = nd.y - by[k], dz = nd.z - bz[k];
                opens += !(dz * dz + (dy * dy + dx * dx) >= nd.rcrit2);
            }
            if (nd.body >= 0) opens = 0;
            const bool every = opens == 0;            /* accepted by every body */
            /* the furthest Next of such an entry up to this lane */
            const int reach = nbh_scan_max(in && every ? nd.next : 0);
            const int before =
                max(skip, __builtin_amdgcn_update_dpp(0, reach, 0x138, 0xF, 0xF, false));
            skip = max(skip, __builtin_amdgcn_readlane(reach, 63));
            const bool keep = in && opens < B && q >= before;
            const unsigned long long km = __builtin_amdgcn_ballot_w64(keep);
            const int at = tail + (int) nbh_mbcnt(km);
            if (keep) rnext[at & (NBH_LIST_RING - 1)] = nd.next;
            nbh_wave_sync();
            if (keep) {
                unsigned cont = 0;
                #pragma unroll
                for (int d = 1; d < S; ++d)
                    if (rnext[(at - d) & (NBH_LIST_RING - 1)] > q) cont |= 1u << (S - d);
                ring[at & (NBH_LIST_RING - 1)] = make_int2(q, (int) cont);
            }
            nbh_wave_sync();
            tail += __popcll(km);
            int left = (tail - head) / S;
            if (!AHEAD) {
                for (; left > 0; --left, head += S) batch(fetch<QUAD>(head, S), S);
            } else if (left > 0) {
                /* two sets of registers; the last fetch may be of stale
                 * entries, whose nodes exist */
                ListRec ra = fetch<QUAD>(head, S);
                for (;;) {
                    const ListRec rb = fetch<QUAD>(head + S, S);
                    batch(ra, S);
                    head += S;
                    if (--left == 0) break;
                    ra = fetch<QUAD>(head + S, S);
                    batch(rb, S);
                    head += S;
                    if (--left == 0) break;
                }
            }
        }
        if (tail > head) batch(fetch<QUAD>(head, tail - head), tail - head);
    }
};

#endif
