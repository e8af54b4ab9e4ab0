/*
 * The event loop of one system on a whole workgroup (gfx950): NW wavefronts
 * handle the next NW events of the calendar at once and commit those that
 * the serial order allows, so the results are those of the loop of one
 * wavefront bit for bit.
 *
 * What bounds that loop for few systems is one wavefront's latency: about
 * 4 microseconds per event of dependent instructions and memory round trips,
 * on a chip whose other wavefront slots are empty.  Events of disks that are
 * not neighbours do not see each other, so the next few can be worked out
 * from the same state.
 *
 * A round, between barriers:
 *   scan     the keys of the calendar nodes below a moving time limit are
 *            gathered from LDS, while the first wavefront brings the loop's
 *            state up to date
 *   order    every wavefront places its share of them among the others, and
 *            marks those that an earlier one takes away (a collision
 *            re-predicts its partner, whose own event, often the same
 *            collision seen from the other disk, then never pops); wavefront w
 *            picks the w-th of the rest
 *   compute  every wavefront works out its event without writing
 *            (event_open, event_predict<SPEC>)
 *   check    every wavefront tests its event against the ones before it: it
 *            must be earlier than anything they leave behind and read no disk
 *            or cell that they write
 *   commit   the longest prefix that the serial loop would handle in the same
 *            way (no failed test, no scheduled event, ring wrap or bound in
 *            it) is written: insertion counters, sums, tape and trace
 *            positions follow from the events' order in it
 * The first event of a round always commits, so the loop advances whatever
 * the limit or the spatial distribution; scheduled events and ring wraps are
 * handled between rounds by the whole workgroup.
 *
 * What a round costs and gives (cycles, and events committed): 400 disks in
 * LDS on 8 wavefronts 16100, 3.7; 512 such systems on 4 wavefronts each 16900,
 * 3.0; 2000 disks on 16 wavefronts 21800, 11.8; 2^20 disks 40800, 13.2; 1000
 * disks in a channel under the field on 8 wavefronts 24300, 4.5.  More than half
 * of the wavefronts' cycles are waits (52 to 65%), for memory and at the
 * barriers.  The scan and the ordering are a part that no event shares: while
 * the first wavefront alone did them, a chain of some thirty dependent LDS
 * accesses, they took 2600 and 4250 of 19000 cycles (2000 disks on 8
 * wavefronts).  Spread over the wavefronts, one comparison of 64 lanes per
 * entry, and with one count for a scan's four nodes a lane, that round went to
 * 17400 (4000 collisions 6.76 ms to 6.20).
 *
 * The calendar's window level lives in LDS: the leaves themselves up to
 * EDMD_WIDE_FLAT disks, else the first level of at most EDMD_WIDE_NODES
 * nodes; the levels above it are made again when the loop ends.
 *
 * Compiled once per variant, as edmd_loop.hip.  Reference line numbers are
 * those of src/EDMD.c.
 */
#define EDMD_DEVICE_ARRAYS 1
#include "edmd_loop.h"
#include "edmd_lds.h"
#include "edmd_variants.h"

namespace {

/* A calendar node below the scan's time limit. */
struct WideEntry {
    double key;
    int64_t rank;
    int32_t p, aux; /* leaf and event code */
};
template <int NW>
constexpr int WIDE_LIST = NW > 8 ? 64 : 32; /* entries an order takes: a lane each */

/* An entry in the order of (time, rank). */
struct WideOrder {
    double key;
    int32_t p, aux;
    int32_t flags; /* WO_*, and from bit 2 the place of the one that takes it away */
    int32_t pad;
};
enum { WO_SHADOWED = 1, WO_STOP = 2 };

/* An event as a wavefront takes it. */
struct WidePick {
    double key, paul; /* its time; bucket start when it is handled */
    int32_t p, aux;
    int32_t steps; /* buckets passed before it in this round */
    int32_t plain; /* 0: no event for this wavefront */
    int32_t ord;   /* its place among the gathered events */
    int32_t shad;  /* place of the first one that it takes away (64: none) */
};

/* A worked-out event, as the others see it. */
struct WideSlot {
    double key;      /* its time */
    double lim;      /* earliest event it leaves behind: new leaves, its group's next leaf */
    int32_t p, j;    /* disks it changes (j = -2: none) */
    int32_t ca, cb;  /* cells of the disks it changes (a crossing: entered, left), x | y << 16 */
    int32_t flags, type;
    int32_t gp, gj;  /* window nodes of its leaves */
    double vir[4];   /* its virial terms */
    double wsum;     /* its term of the tape's virial sum */
    double ax, ay, cx, cy, ff; /* its tape record's */
    double dp[4];    /* its momentum to the walls */
};

enum { WS_COLL = 1, WS_WALL = 2, WS_OV = 4, WS_FULL = 8 };

/* A wavefront's word of the round's verdict. */
enum {
    WB_OK = 1, WB_LAST = 2, WB_COUNTED = 4, WB_TAPED = 8, WB_INS = 16, WB_SHARE = 128,
    WB_CROSS = 256
};

/* The nodes above an event's new leaves up to the window level (in LDS
 * until the event commits). */
struct PathNodes {
    double kA[2], kB[2];
    int iA[2], iB[2], xA[2], xB[2];
    int64_t rA, rB; /* of the window level's */
};

/* What the leader decides. */
enum { WT_ROUND, WT_SCAN, WT_SPECIAL, WT_WRAP, WT_STOP };

/* The loop's state, the leader's: in LDS between its parts of a round, so
 * that it costs the events no registers. */
struct WideState {
    LoopRegs R;
    uint64_t ncross;
    int64_t ntape, ntrace;
    double width; /* of the window */
    int32_t last_type, guard, tries, reason;
    int32_t halt; /* a kind of event that stops the run was handled */
};

template <int NW>
struct WideShared {
    int32_t cand[NW][EDMD_STAGE_MAX];
    WideState state;
    WidePick pick[NW];
    WideSlot slot[NW];
    PathNodes nodes[NW];
    WideEntry list[WIDE_LIST<NW>];
    WideOrder sorted[WIDE_LIST<NW>];
    int32_t verdict[NW];
    int32_t lcount, todo, cut, sums, moved; /* cut: events the last round committed */
    int32_t given; /* the list is wide_first's, not the scan's */
    int32_t stop; /* why the loop stops, EDMD_STOP_NONE: it goes on */
    int32_t room, croom; /* events and counted events that the bounds leave */
    double lim;          /* the scan's time limit */
    double vir[4];
    double red[2];
    int64_t ctr, ntape, ntrace;
    int64_t ev_limit; /* the run's */
    uint64_t coll_limit;
};

/* The calendar's window level in LDS (SoA: the search reads keys alone). */
struct WideCal {
    double EDMD_LDS* key;
    int64_t EDMD_LDS* rank; /* of the node's leaf */
    int32_t EDMD_LDS* aux;
    int32_t EDMD_LDS* idx; /* leaf of a node; window of leaves: unused */
    int ls;                /* level */
    int m;                 /* nodes */
};

/* The ranks of a window of leaves are the leaves' own: where the arrays are in
 * LDS they are not kept twice.  So two systems of 400 disks fit a CU (80 KB
 * each, 83 with the copy): 512 of them, 4000 collisions, 15.1 ms from HBM, 13.8
 * from LDS. */
__device__ __forceinline__ constexpr bool ranks_apart(const EdmdArrays&) { return true; }
__device__ __forceinline__ constexpr bool ranks_apart(const EdmdArraysL&) { return false; }
__device__ __forceinline__ int64_t EDMD_LDS* window_ranks(const EdmdArrays&,
                                                          unsigned char EDMD_LDS* apart) {
    return (int64_t EDMD_LDS*)apart;
}
__device__ __forceinline__ int64_t EDMD_LDS* window_ranks(const EdmdArraysL& A,
                                                          unsigned char EDMD_LDS*) {
    return A.lrank;
}

/* Waits for this wavefront's LDS accesses only, then for the others: memory
 * writes stay in flight. */
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <class AR>
__device__ __forceinline__ void cal_put(const WideCal& W, int node, double key, int64_t rank,
                                        int leaf, int aux) {
    W.key[node] = key;
    W.rank[node] = rank;
    W.aux[node] = aux;
    if (W.ls > 0) W.idx[node] = leaf;
}

/* Makes the window level from the leaves (and the levels between). */
template <int NT, class AR>
__device__ void cal_build(const EdmdConst& C, const AR& A, const WideCal& Wc, int tid) {
    for (int l = 1; l <= Wc.ls; ++l) {
        for (int g = tid; g < C.lsize[l]; g += NT) node_min(C, A, l, g);
        __syncthreads();
    }
    const auto nd = level(A, Wc.ls);
    for (int g = tid; g < Wc.m; g += NT) {
        const EdmdNode n = nd[g];
        cal_put<AR>(Wc, g, n.key, A.lrank[n.idx], n.idx, n.aux);
    }
    __syncthreads();
}

/* Writes the window level back and makes the levels above it again. */
template <int NT, class AR>
__device__ void cal_close(const EdmdConst& C, const AR& A, const WideCal& Wc, int tid) {
    if (Wc.ls > 0) {
        const auto nd = level(A, Wc.ls);
        for (int g = tid; g < Wc.m; g += NT) {
            EdmdNode n;
            n.key = Wc.key[g];
            n.idx = Wc.idx[g];
            n.aux = Wc.aux[g];
            nd[g] = n;
        }
    }
    __syncthreads();
    for (int l = Wc.ls + 1; l <= C.nlev; ++l) {
        for (int g = tid; g < C.lsize[l]; g += NT) node_min(C, A, l, g);
        __syncthreads();
    }
}

/* Minimum of one node's 64 children, held one per lane, by (key, rank), with
 * the winner's rank.  The ranks of the event's own new leaves are taken with
 * the insertion counter of the round's start: they compare with the stored
 * ones as the final ones will (a new direct rank is above every stored one, a
 * new bucket rank below). */
__device__ __forceinline__ void group_min(int lane, double& k, int& i, int& x, int64_t& r) {
    const double mk = wave_min(k);
    const uint64_t at = __ballot(k == mk);
    int w = (int)__builtin_ctzll(at);
    if (__popcll(at) > 1 && mk < INF_D) {
        const bool tie = lane_in(at);
        int64_t q = tie ? r : INT64_MAX;
        int l = tie ? lane : 64;
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const long long oq = __shfl_xor((long long)q, m, 64);
            const int ol = __shfl_xor(l, m, 64);
            if (oq < q || (oq == q && ol < l)) {
                q = oq;
                l = ol;
            }
        }
        w = __builtin_amdgcn_readfirstlane(l);
    }
    k = mk;
    i = __builtin_amdgcn_readlane(i, w);
    x = __builtin_amdgcn_readlane(x, w);
    r = lane_value64(r, w);
}

__device__ __forceinline__ bool cells_near(int a, int b, int reach, int ncx, int ncy) {
    int dx = (a & 0xffff) - (b & 0xffff);
    int dy = (a >> 16) - (b >> 16);
    dx = dx < 0 ? -dx : dx;
    dy = dy < 0 ? -dy : dy;
    return (dx <= reach || dx >= ncx - reach) && (dy <= reach || dy >= ncy - reach);
}

/* The children, with their ranks, on the paths of leaves pA and pB (pB < 0:
 * none) up to the window level ls (1 or 2). */
struct PathWindow {
    double k[2][2];
    int i[2][2], x[2][2];
    int64_t r[2][2];
};

template <class AR>
__device__ __forceinline__ void path_window(const EdmdConst& C, const AR& A, int lane, int ls,
                                            int pA, int pB, PathWindow& P) {
#pragma unroll
    for (int l = 0; l < 2; ++l) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int p = h ? pB : pA;
            double k = INF_D;
            int i = 0, x = 0;
            int64_t r = 0;
            if (l < ls && p >= 0) {
                const int c = ((p >> (6 * (l + 1))) << 6) + lane;
                if (c < C.lsize[l]) {
                    const EdmdNode nd = level(A, l)[c];
                    k = nd.key;
                    i = nd.idx;
                    x = nd.aux;
                    if (l == 0) r = A.lrank[c];
                }
            }
            P.k[h][l] = k;
            P.i[h][l] = i;
            P.x[h][l] = x;
            P.r[h][l] = r;
        }
    }
}

template <class AR>
__device__ __forceinline__ void path_nodes(const AR& A, int lane, int ls, PathWindow& P, int pA,
                                           double kA, int xA, int64_t rA, int pB, double kB,
                                           int xB, int64_t rB, PathNodes& N, double& limA,
                                           double& limB) {
    int iA = pA, iB = pB, cA = pA, cB = pB;
#pragma unroll
    for (int l = 0; l < 2; ++l) {
        if (l >= ls) break;
        if (l == 1) {
            P.r[0][1] = A.lrank[P.i[0][1]];
            P.r[1][1] = A.lrank[P.i[1][1]];
        }
        const int gA = cA >> 6, gB = pB >= 0 ? cB >> 6 : -1;
        const int c = (gA << 6) + lane;
        const bool a = c == cA, b = pB >= 0 && c == cB;
        double k = a ? kA : (b ? kB : P.k[0][l]);
        int i = a ? iA : (b ? iB : P.i[0][l]), x = a ? xA : (b ? xB : P.x[0][l]);
        int64_t r = a ? rA : (b ? rB : P.r[0][l]);
        group_min(lane, k, i, x, r);
        double k2 = k;
        int i2 = i, x2 = x;
        int64_t r2 = r;
        if (pB >= 0 && gB != gA) {
            const bool o = (gB << 6) + lane == cB;
            k2 = o ? kB : P.k[1][l];
            i2 = o ? iB : P.i[1][l];
            x2 = o ? xB : P.x[1][l];
            r2 = o ? rB : P.r[1][l];
            group_min(lane, k2, i2, x2, r2);
        }
        kA = k;
        iA = i;
        xA = x;
        kB = k2;
        iB = i2;
        xB = x2;
        if (lane == 0) {
            N.kA[l] = k;
            N.iA[l] = i;
            N.xA[l] = x;
            N.kB[l] = k2;
            N.iB[l] = i2;
            N.xB[l] = x2;
        }
        rA = r;
        rB = r2;
        cA = gA;
        cB = gB;
    }
    if (lane == 0) {
        N.rA = rA;
        N.rB = rB;
    }
    limA = kA;
    limB = kB;
}

template <class AR>
__device__ __forceinline__ void node_put(const AR& A, const WideCal& Wc, int l, int g, double key,
                                         int64_t rank, int leaf, int aux) {
    if (l == Wc.ls) {
        cal_put<AR>(Wc, g, key, rank, leaf, aux);
    } else {
        EdmdNode n;
        n.key = key;
        n.idx = leaf;
        n.aux = aux;
        A.lev[l - 1][g] = n;
    }
}

/* The final ranks of the event's own leaves, where they are a node's. */
template <class AR>
__device__ __forceinline__ void nodes_store(const AR& A, const WideCal& Wc, int pA, int64_t rkA,
                                            int pB, int64_t rkB, const PathNodes& N) {
    auto rank = [&](int leaf, int64_t r) { return leaf == pA ? rkA : (leaf == pB ? rkB : r); };
#pragma unroll
    for (int l = 1; l <= 2; ++l) {
        if (l > Wc.ls) break;
        const int gA = pA >> (6 * l), gB = pB >= 0 ? pB >> (6 * l) : gA;
        node_put(A, Wc, l, gA, N.kA[l - 1], rank(N.iA[l - 1], N.rA), N.iA[l - 1], N.xA[l - 1]);
        if (gB != gA)
            node_put(A, Wc, l, gB, N.kB[l - 1], rank(N.iB[l - 1], N.rB), N.iB[l - 1], N.xB[l - 1]);
    }
}

/* The node of level l above leaf p, from its children in memory. */
template <class AR>
__device__ __forceinline__ void node_make(const EdmdConst& C, const AR& A, const WideCal& Wc,
                                          int lane, int l, int p, double base) {
    const int g = p >> (6 * l), c = (g << 6) + lane;
    double k = INF_D;
    int i = 0x7fffffff, x = 0;
    if (c < C.lsize[l - 1]) {
        const EdmdNode nd = level(A, l - 1)[c];
        k = nd.key;
        i = nd.idx;
        x = nd.aux;
    }
    wave_argmin(A, base, k, i, x);
    if (lane == 0) node_put(A, Wc, l, g, k, A.lrank[k < INF_D ? i : 0], i, x);
}

/* The overflow list filed again at a wrap of the bucket ring (refile_wrap's
 * steps, EDMD.c:2292-2302) by the whole workgroup; moved: whether any leaf
 * was made again. */
template <int NT, class AR>
__device__ void wide_refile(const EdmdConst& C, const AR& A, int tid, double paul, int64_t win,
                            int64_t& ctr, int32_t* moved, int64_t* shared_ctr) {
    if (tid < 64) {
        int64_t c = ctr;
        refile_specials(C, A.st, paul, win, c);
        if (tid == 0) {
            *shared_ctr = c;
            *moved = 0;
        }
    }
    __syncthreads();
    const int64_t now = *shared_ctr, lo = A.st->ovf_lo;
    bool any = false;
    for (int k = tid; k < C.n; k += NT) any |= refile_disk(C, A, k, paul, now);
    if (any) *moved = 1;
    __syncthreads();
    if (tid == 0) A.st->ovf_lo = now;
    ctr = 2 * now - lo;
    __syncthreads();
}

/* The neighbours' flights under the field or damping (EDMD.c:2664-2666) of a
 * committed event, after its own records are stored: the candidates are
 * still staged. */
template <class AR>
__device__ __forceinline__ void fly_neighbours(const EdmdConst& C, const AR& A, int lane, double t,
                                               const EvState& S, const int32_t* stage) {
    const bool two = S.nown == 2, hi = lane >= 32;
    const int32_t* const st = stage + ((two && hi) ? EDMD_STAGE_HALF : 0) + EDMD_STAGE_CAP;
    const int n = (two && hi) ? S.totB : S.totA;
    const int most = S.totA > S.totB ? S.totA : S.totB;
    const int step = two ? 32 : 64;
    for (int base = 0; base < most; base += step) {
        const int f = base + (two ? (lane & 31) : lane);
        const int q = f < n ? st[f] : -1;
        if (q >= 0 && q != S.own) {
            EdmdPart r = A.p[q];
            fly_v<true>(C, t, r.x, r.y, r.vx, r.vy, r.tl);
            const auto w = A.p + q;
            w->x = r.x;
            w->y = r.y;
            w->vx = r.vx;
            w->vy = r.vy;
            w->tl = r.tl;
        }
    }
}

/* This wavefront's share of the n gathered nodes, entries wave, wave + NW, ...:
 * each one's place by (time, rank) and whether an earlier one takes it away.
 * Every lane holds an entry, so one comparison a lane places one of them. */
template <int NW>
__device__ __forceinline__ void wide_rank(WideShared<NW>& Sh, int lane, int wave, int n) {
    const bool in = lane < n;
    const WideEntry me = Sh.list[in ? lane : 0];
    const double key = in ? me.key : INF_D;
    const int p = in ? me.p : -1, aux = in ? me.aux : -1;
    const int64_t rank = me.rank;
    /* the entries before e, and those whose partner e's disk is */
    auto look = [&](int e, uint64_t& sooner, uint64_t& hit) {
        const double ke = lane_value(key, e);
        const int64_t re = lane_value64(rank, e);
        sooner = __ballot((key < ke) | (in & (key == ke) & (rank < re)));
        hit = __ballot(aux == __builtin_amdgcn_readlane(p, e));
    };
    for (int e = wave; e < n; e += NW) {
        uint64_t sooner, hit;
        look(e, sooner, hit);
        const int place = (int)__popcll(sooner);
        int flags = 0;
        if (hit) {
            /* taken away by entry `by`, if that comes earlier; where it is
             * itself taken away, or several name this disk, the window ends
             * here */
            const int by = 63 - (int)__builtin_clzll(hit);
            const bool shadowed = ((sooner >> by) & 1) != 0;
            bool stop = __popcll(hit) > 1 && place > 0;
            if (shadowed) {
                uint64_t bsooner, bhit;
                look(by, bsooner, bhit);
                if (bhit) stop |= ((bsooner >> (63 - (int)__builtin_clzll(bhit))) & 1) != 0;
                flags = WO_SHADOWED | ((int)__popcll(bsooner) << 2);
            }
            if (stop) flags |= WO_STOP;
        }
        if (lane == e) {
            WideOrder& o = Sh.sorted[place];
            o.key = key;
            o.p = p;
            o.aux = aux;
            o.flags = flags;
        }
    }
}

/* The buckets up to an event at `key` (pick_next): paul and steps; whether it
 * is a plain one, not behind a ring wrap or a scheduled event. */
__device__ __forceinline__ bool wide_buckets(const EdmdConst& C, const LoopRegs& R, bool on,
                                             double key, double& paul, int& steps) {
    paul = R.paul;
    steps = 0;
    const int cur = R.cur;
    const int64_t win = R.win, swin = R.swin;
    bool plain = on && key < INF_D && key < R.next_special && !(swin >= 0 && swin <= win);
    while (plain && !(key - paul < C.dtp)) {
        paul = paul + C.dtp;
        ++steps;
        if (cur + steps >= C.nlists || steps > 4096 || (swin >= 0 && swin <= win + steps))
            plain = false;
    }
    return plain;
}

/* This wavefront's event of the n ordered ones, into its pick and k; false
 * where the earliest one is not plain. */
template <int NW, bool W>
__device__ __forceinline__ bool wide_pick(const EdmdConst& C, WideShared<NW>& Sh, int lane,
                                          int wave, int n, WidePick& k) {
    const WideOrder me = Sh.sorted[lane < n ? lane : 0];
    const int flags = lane < n ? me.flags : 0;
    uint64_t use = __ballot(lane < n && !(flags & WO_SHADOWED));
    const uint64_t end = __ballot((flags & WO_STOP) != 0);
    if (end) use &= ((uint64_t)1 << __builtin_ctzll(end)) - 1;
    const uint64_t mine = __ballot(lanes_before(use) == wave && lane_in(use));
    const int ord = mine ? (int)__builtin_ctzll(mine) : 0;
    double paul;
    int steps;
    const bool plain = wide_buckets(C, Sh.state.R, lane == 0 || lane == ord, me.key, paul, steps);
    const uint64_t plains = __ballot(plain);
    k.key = lane_value(me.key, ord);
    k.paul = lane_value(paul, ord);
    k.p = __builtin_amdgcn_readlane(me.p, ord);
    k.aux = __builtin_amdgcn_readlane(me.aux, ord);
    k.steps = __builtin_amdgcn_readlane(steps, ord);
    k.ord = ord;
    const uint64_t takes = __ballot((flags & WO_SHADOWED) != 0 && (flags >> 2) == ord);
    k.shad = takes ? (int)__builtin_ctzll(takes) : 64;
    k.plain = mine && ((plains >> ord) & 1) ? 1 : 0;
    if (W && C.thermal_wall && wave > 0 && k.aux <= EDMD_WALL_CODE(0)) k.plain = 0;
    if (lane == 0) Sh.pick[wave] = k;
    return (plains & 1) != 0;
}

/* The earliest nodes, where the window held more than the list takes (by the
 * leader): every lane's earliest one before which no lane has a second.  A limit
 * in time does not part nodes at one time: with one drawn again and again, then
 * one event a round, the first 8000 events of 2000 disks on a lattice (some on
 * their cells' edges, which they cross at time 0) took 1.9 us each, now 1.1; a
 * front of 4096 disks at one speed 22 us, now 14, for its events in turn lie
 * beside one another (one wavefront: 5.2). */
template <int NW>
__device__ __forceinline__ void wide_first(const WideCal& Wc, WideShared<NW>& Sh, int lane) {
    double k1 = INF_D, k2 = INF_D;
    int64_t r1 = 0, r2 = 0;
    int node = -1;
    if (lane < WIDE_LIST<NW>) {
        for (int g = lane; g < Wc.m; g += WIDE_LIST<NW>) {
            const double k = Wc.key[g];
            if (!(k < INF_D && k <= k2)) continue;
            const int64_t r = Wc.rank[g];
            if (k < k1 || (k == k1 && r < r1)) {
                k2 = k1;
                r2 = r1;
                k1 = k;
                r1 = r;
                node = g;
            } else if (k < k2 || r < r2) {
                k2 = k;
                r2 = r;
            }
        }
    }
    const double kt = wave_min(k2);
    long long rt = k2 == kt ? r2 : INT64_MAX;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        const long long o = __shfl_xor(rt, m, 64);
        rt = o < rt ? o : rt;
    }
    const bool in = node >= 0 && (k1 < kt || (k1 == kt && r1 < rt));
    const uint64_t all = __ballot(in);
    if (in) {
        WideEntry e;
        e.key = k1;
        e.rank = r1;
        e.p = Wc.ls > 0 ? Wc.idx[node] : node;
        e.aux = Wc.aux[node];
        Sh.list[lanes_before(all)] = e;
    }
    const double k0 = wave_min(k1);
    WAVE_SYNC();
    if (lane == 0) {
        if (kt > k0) Sh.state.width *= 0.5;
        Sh.lcount = (int)__popcll(all);
        Sh.given = 1;
        Sh.lim = -INF_D; /* the scan adds none */
    }
}

/* The leader's decision where a round cannot start from the gathered nodes:
 * too many of them (the first of them, WT_SCAN) or none (another limit,
 * WT_SCAN; the earliest event alone after twelve), or the earliest one is not
 * plain (what findNextEvent does next, EDMD.c:2313-2327, one ring wrap at a
 * time). */
template <int NW, class AR>
__device__ __forceinline__ int wide_decide(const EdmdConst& C, const AR& A, int lane,
                                           const WideCal& Wc, WideShared<NW>& Sh, bool ordered) {
    WideState& Z = Sh.state;
    LoopRegs& R = Z.R;
    double width = Z.width;
    if (!ordered && Sh.lcount > WIDE_LIST<NW>) {
        wide_first<NW>(Wc, Sh, lane);
        return WT_SCAN;
    }
    if (!ordered && Z.tries < 12) {
        width *= 4.0;
        WAVE_SYNC();
        if (lane == 0) {
            ++Z.tries;
            Z.width = width;
            Sh.lcount = 0;
            Sh.lim = R.t + width;
        }
        return WT_SCAN;
    }
    double k0 = INF_D;
    int64_t rank = 0;
    int node = 0;
    for (int g = lane; g < Wc.m; g += 64) {
        const double k = Wc.key[g];
        if (k < k0 || (k == k0 && k < INF_D && Wc.rank[g] < rank)) {
            k0 = k;
            rank = Wc.rank[g];
            node = g;
        }
    }
    int leaf = Wc.ls > 0 ? Wc.idx[node] : node, who = lane;
    wave_argmin(A, R.t, k0, leaf, who);
    node = __builtin_amdgcn_readlane(node, who);
    const int p0 = Wc.ls > 0 ? Wc.idx[node] : node, aux0 = Wc.aux[node];
    if (lane == 0) {
        Z.tries = 0;
        Sh.lcount = 0;
        Sh.lim = k0 + width;
    }
    WAVE_SYNC();
    if (!(k0 < INF_D) && !(R.next_special < INF_D)) {
        if (lane == 0) Z.reason = EDMD_STOP_EMPTY;
        return WT_STOP;
    }
    double paul;
    int steps;
    if (!wide_buckets(C, R, true, k0, paul, steps)) {
        double rpaul = R.paul;
        int64_t win = R.win;
        int cur = R.cur, guard = Z.guard, todo = -1;
        for (;; ++guard) {
            const bool part_in = k0 - rpaul < C.dtp;
            const bool spec_in = R.swin >= 0 && R.swin <= win;
            auto sooner = [&]() {
                return before(R.next_special, R.srank, k0,
                              k0 == R.next_special ? uni64(A.lrank[p0]) : (int64_t)0);
            };
            bool special;
            if (part_in || spec_in) {
                special = spec_in && (!part_in || sooner());
            } else if (!(k0 < 1e25) && !(R.next_special < 1e25)) {
                special = R.next_special <= k0;
            } else if (guard >= (1 << 24)) {
                const double tn = k0 < R.next_special ? k0 : R.next_special;
                while (!(tn - rpaul < C.dtp)) {
                    rpaul = rpaul + C.dtp;
                    win++;
                }
                special = sooner();
            } else {
                rpaul = rpaul + C.dtp;
                win++;
                if (++cur >= C.nlists) {
                    cur = 0;
                    ++guard;
                    todo = WT_WRAP;
                    break;
                }
                continue;
            }
            if (special) todo = WT_SPECIAL;
            break;
        }
        WAVE_SYNC();
        if (lane == 0) {
            R.paul = rpaul;
            R.win = win;
            R.cur = cur;
            Z.guard = guard;
        }
        if (todo >= 0) return todo;
        /* a particle event after all, alone */
        paul = rpaul;
        steps = 0;
    }
    if (lane < NW) {
        WidePick k;
        k.key = k0;
        k.paul = paul;
        k.p = p0;
        k.aux = aux0;
        k.steps = steps;
        k.plain = lane == 0 ? 1 : 0;
        k.ord = 0;
        k.shad = 64;
        Sh.pick[lane] = k;
    }
    return WT_ROUND;
}

/* The round's verdict: one bit a wavefront each. */
struct WideVerdict {
    uint32_t ok, last, counted, taped, one, two, four, share, cross;
};

template <int NW>
__device__ __forceinline__ WideVerdict wide_verdict(const WideShared<NW>& Sh, int lane) {
    const int v = lane < NW ? Sh.verdict[lane] : 0;
    WideVerdict V;
    V.ok = (uint32_t)__ballot((v & WB_OK) != 0);
    V.last = (uint32_t)__ballot((v & WB_LAST) != 0);
    V.counted = (uint32_t)__ballot((v & WB_COUNTED) != 0);
    V.taped = (uint32_t)__ballot((v & WB_TAPED) != 0);
    V.one = (uint32_t)__ballot((v & WB_INS) != 0);
    V.two = (uint32_t)__ballot((v & (2 * WB_INS)) != 0);
    V.four = (uint32_t)__ballot((v & (4 * WB_INS)) != 0);
    V.share = (uint32_t)__ballot((v & WB_SHARE) != 0);
    V.cross = (uint32_t)__ballot((v & WB_CROSS) != 0);
    return V;
}

/* The events of a round that commit: up to the first one that failed its
 * test, the first after which the loop stops, the bounds. */
template <int NW>
__device__ __forceinline__ int wide_cut(const WideVerdict& V, int room, int croom) {
    int cut = (int)__builtin_ctz(~V.ok | (1u << NW));
    if (V.last) {
        const int c = (int)__builtin_ctz(V.last) + 1;
        cut = c < cut ? c : cut;
    }
    cut = room < cut ? room : cut;
    if (croom <= NW) {
        int c = 0, m = 0;
        for (; m < cut && c < croom; ++m) c += (int)(V.counted >> m) & 1;
        cut = m;
    }
    return cut;
}

/* Insertions of the events below m. */
__device__ __forceinline__ int wide_inserts(const WideVerdict& V, int m) {
    const uint32_t below = (1u << m) - 1;
    return __popc(V.one & below) + 2 * __popc(V.two & below) + 4 * __popc(V.four & below);
}

/* The loop's state after a round of `cut` events (the leader), what the next
 * round needs of it, and whether there is one. */
template <int NW>
__device__ __forceinline__ void wide_advance(const EdmdConst& C, WideShared<NW>& Sh, int lane,
                                             const EdmdRunArgs& ra) {
    WideState& Z = Sh.state;
    LoopRegs& R = Z.R;
    const int cut = __builtin_amdgcn_readfirstlane(Sh.cut); /* 0: no round since */
    const WideVerdict V = wide_verdict<NW>(Sh, lane);
    if (lane != 0) return;
    double t = R.t;
    int64_t ctr = R.ctr, ntape = Z.ntape, ntrace = Z.ntrace, nevents = (int64_t)R.nevents;
    uint64_t ncol = R.ncol;
    int status = R.status, halt = Z.halt;
    if (cut > 0) {
        const uint32_t done = (1u << cut) - 1;
        const WideSlot& last = Sh.slot[cut - 1];
        const WidePick& lp = Sh.pick[cut - 1];
        const int type = last.type, flags = last.flags;
        t = lp.key;
        ctr += wide_inserts(V, cut);
        ncol += (uint64_t)__popc(V.counted & done);
        nevents += cut;
        if (C.trace_cap > 0) ntrace += cut;
        ntape += __popc(V.taped & done);
        if (ra.stop_mask & (1 << type)) halt = 1;
        if (flags & WS_FULL) {
            status = EDMD_DEV_CELL_OVERFLOW;
            R.err_i = last.p;
            R.err_j = (last.ca >> 16) * C.ncx + (last.ca & 0xffff);
            ctr -= 2; /* the crossing stops before its insertions */
        } else if (flags & WS_OV) {
            status = EDMD_DEV_OVERLAP;
            R.err_i = last.p;
        }
        R.t = t;
        R.paul = lp.paul;
        R.win += lp.steps;
        R.cur += lp.steps;
        R.ncol = ncol;
        R.nevents = (uint64_t)nevents;
        R.status = status;
        R.ctr = ctr;
        Z.last_type = type;
        Z.ntape = ntape;
        Z.ntrace = ntrace;
        Z.ncross += (uint64_t)__popc(V.cross & done);
        Z.guard = 0;
        Z.halt = halt;
    }
    const int64_t ev_limit = Sh.ev_limit, er = ev_limit - nevents;
    const uint64_t coll_limit = Sh.coll_limit;
    const uint64_t cr = coll_limit - ncol;
    Sh.room = er < NW ? (int)er : NW;
    Sh.croom = cr <= NW ? (int)cr : NW + 1;
    Sh.ctr = ctr;
    Sh.ntape = ntape;
    Sh.ntrace = ntrace;
    int why = EDMD_STOP_NONE;
    if (halt) why = EDMD_STOP_SPECIAL;
    else if (status != EDMD_DEV_OK) why = EDMD_STOP_ERROR;
    else if (nevents >= ev_limit) why = EDMD_STOP_EVENTS;
    else if (ncol >= coll_limit) why = EDMD_STOP_COLLISIONS;
    else if (!(t <= ra.tmax)) why = EDMD_STOP_TIME;
    Sh.stop = why;
    if (why != EDMD_STOP_NONE) Z.reason = why;
}

template <int NW, bool FLAT, bool G, bool W, class AR>
__device__ __forceinline__ void wide_loop(const EdmdConst& Cs, const AR& As, EdmdRunArgs ra,
                                          unsigned char EDMD_LDS* pool) {
    constexpr int NT = 64 * NW;
    static_assert(NW <= 16, "a bit of the verdict's masks per wavefront");
    __shared__ WideShared<NW> Sh;
    const int tid0 = threadIdx.x;
    int tid = tid0, lane = tid & 63, wave = wave_in_group();
    WideCal Wc;
    {
        const EdmdConst& C = opaque(Cs);
        const AR& A = opaque(As);
        const EdmdState* st = A.st;
        Wc.ls = FLAT ? 0 : edmd_wide_level(&C);
        Wc.m = C.lsize[Wc.ls];
        Wc.key = (double EDMD_LDS*)pool;
        Wc.rank = window_ranks(A, pool + (size_t)Wc.m * 8);
        Wc.aux = (int32_t EDMD_LDS*)(pool + (size_t)Wc.m * (ranks_apart(A) ? 16 : 8));
        Wc.idx = Wc.aux + Wc.m;
        WideState Z;
        LoopRegs& R = Z.R;
        R.q = nullptr;
        R.t = st->t;
        R.ncol = st->ncol;
        R.nevents = st->nevents;
        R.status = st->status;
        R.err_i = st->err_i;
        R.err_j = st->err_j;
        R.paul = st->paul;
        R.ctr = st->ctr;
        R.win = st->win;
        R.cur = (int)(R.win % C.nlists);
        next_special(st, R);
        Z.ncross = st->ncross;
        Z.last_type = st->last_type;
        Z.ntape = st->ntape;
        Z.ntrace = st->ntrace;
        Z.width = 0.25 / C.n; /* about a window's events; it adapts */
        Z.guard = Z.tries = Z.halt = 0;
        Z.reason = EDMD_STOP_NONE;
        if (tid < 4) Sh.vir[tid] = st->vir[tid];
        if (tid < NW) Sh.verdict[tid] = 0;
        if (tid == 0) {
            Sh.state = Z;
            Sh.ev_limit = st->ev_limit < ra.max_events ? st->ev_limit : ra.max_events;
            Sh.coll_limit = st->coll_limit < ra.max_coll ? st->coll_limit : ra.max_coll;
            Sh.cut = 0;
            Sh.lcount = 0;
            Sh.sums = 0;
            Sh.given = 0;
            Sh.lim = R.t + Z.width;
        }
        cal_build<NT>(C, A, Wc, tid);
    }
    for (;;) {
        int todo;
        {
            for (;;) {
                const EdmdConst& C = opaque(Cs);
                const AR& A = opaque(As);
                /* what follows from the thread or the system's record alone is
                 * made or read again each round, not held in registers */
                asm volatile("" : "+v"(tid), "+v"(lane), "+s"(wave));
                /* scan (the others), the state after the last round (the
                 * leader) */
                if (wave == 0) {
                    wide_advance<NW>(C, Sh, lane, ra);
                } else {
                    const double lim = Sh.lim;
                    for (int g0 = tid - 64; g0 - lane < Wc.m; g0 += 4 * (NT - 64)) {
                        double k[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const int g = g0 + u * (NT - 64);
                            k[u] = g < Wc.m ? Wc.key[g] : INF_D;
                        }
                        const double least = min_f64(min_f64(k[0], k[1]), min_f64(k[2], k[3]));
                        if (!__ballot(least < lim)) continue;
                        /* one count for the four */
                        int all = 0;
#pragma unroll
                        for (int u = 0; u < 4; ++u) all += (int)__popcll(__ballot(k[u] < lim));
                        int at = 0;
                        if (lane == 0) at = atomicAdd(&Sh.lcount, all);
                        at = __builtin_amdgcn_readfirstlane(at);
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const uint64_t in = __ballot(k[u] < lim);
                            const int to = at + lanes_before(in);
                            at += (int)__popcll(in);
                            if (k[u] < lim && to < WIDE_LIST<NW>) {
                                const int g = g0 + u * (NT - 64);
                                WideEntry e;
                                e.key = k[u];
                                e.rank = Wc.rank[g];
                                e.p = Wc.ls > 0 ? Wc.idx[g] : g;
                                e.aux = Wc.aux[g];
                                Sh.list[to] = e;
                            }
                        }
                    }
                }
                __syncthreads();
                if (wave == NW - 1 && !G) {
                    EdmdState* st = A.st;
                    /* the last round's sums, in its events' order */
                    const int cut = Sh.sums;
                    if (lane < 4) {
                        double u[NW];
                        int f[NW];
#pragma unroll
                        for (int m = 0; m < NW; ++m) {
                            u[m] = Sh.slot[m].vir[lane];
                            f[m] = Sh.slot[m].flags;
                        }
                        double v = Sh.vir[lane];
#pragma unroll
                        for (int m = 0; m < NW; ++m)
                            if (m < cut && (f[m] & WS_COLL)) v += u[m];
                        Sh.vir[lane] = v;
                    }
                    if (lane == 0) {
                        if (C.tape_cap > 0 || (W && C.walls)) {
                            for (int m = 0; m < cut; ++m) {
                                const WideSlot& sm = Sh.slot[m];
                                if (sm.flags & WS_COLL) {
                                    if (C.tape_cap > 0) {
                                        st->wsum += sm.wsum;
                                        st->tlast = sm.key;
                                    }
                                } else if (W && (sm.flags & WS_WALL)) {
                                    st->dpw += sm.dp[0];
                                    if (C.walls & 8) {
                                        st->dpl += sm.dp[1];
                                        st->dpm += sm.dp[2];
                                        st->dpr += sm.dp[3];
                                    }
                                }
                            }
                        }
                        Sh.sums = 0;
                    }
                }
                if (__builtin_amdgcn_readfirstlane(Sh.stop) != EDMD_STOP_NONE) {
                    todo = WT_STOP;
                    break;
                }
                /* order */
                const int n = __builtin_amdgcn_readfirstlane(Sh.lcount);
                const bool listed = n >= 1 && n <= WIDE_LIST<NW>;
                WidePick my;
                bool plain0 = false;
                if (listed) {
                    wide_rank<NW>(Sh, lane, wave, n);
                    lds_barrier();
                    plain0 = wide_pick<NW, W>(C, Sh, lane, wave, n, my);
                    if (tid == 0) {
                        /* the next window: about two nodes a wavefront */
                        const double width = Sh.state.width;
                        if (Sh.given) Sh.given = 0;
                        else if (n < NW + NW / 2) Sh.state.width = width * 1.2 + 1e-300;
                        else if (n > 2 * NW + NW / 4) Sh.state.width = width * 0.85;
                        Sh.state.tries = 0;
                        Sh.lcount = 0;
                    }
                }
                if (!plain0) {
                    lds_barrier(); /* the picks and the count read by all */
                    if (wave == 0) {
                        const int td = wide_decide<NW>(C, A, lane, Wc, Sh, listed);
                        if (lane == 0) Sh.todo = td;
                    }
                    lds_barrier();
                    todo = __builtin_amdgcn_readfirstlane(Sh.todo);
                    if (todo == WT_SCAN) {
                        if (tid == 0) Sh.cut = 0;
                        continue;
                    }
                    if (todo != WT_ROUND) break;
                    my = Sh.pick[wave];
                }

                /* compute */
                EvState S;
                int brief = 0, cellA = 0, cellB = 0, pj2 = -1;
                if (my.plain) {
                    const double t = my.key;
                    const int p = my.p, aux = my.aux;
                    event_open<G, W>(C, A, lane, t, p, aux, S);
                    if (!G && S.kind == EVK_COLLISION) {
                        /* what only the sums and the tape need waits in LDS */
                        WideSlot& me = Sh.slot[wave];
                        if (lane < 4) {
                            const double u = (lane & 1) == 0 ? S.dx : S.dy;
                            const double v = (lane == 0 || lane == 3) ? S.dx : S.dy;
                            me.vir[lane] = S.w * u * v;
                        }
                        if (lane == 0 && C.tape_cap > 0) {
                            me.wsum = S.w * (S.dx * S.dx + S.dy * S.dy);
                            me.ax = S.dx;
                            me.ay = S.dy;
                            me.cx = S.dvx;
                            me.cy = S.dvy;
                            me.ff = S.ff;
                        }
                    }
                    PathWindow P;
                    const int pj = S.nown == 2 ? aux : -1;
                    if (NW <= 8 && Wc.ls > 0) path_window(C, A, lane, Wc.ls, p, pj, P);
                    event_predict<G, W, true>(C, A, lane, t, S, Sh.cand[wave]);
                    /* (16 wavefronts hide its latency and have no registers for it) */
                    if (NW > 8 && Wc.ls > 0) path_window(C, A, lane, Wc.ls, p, pj, P);
                    /* the leaf's key and code do not depend on the counter:
                     * the ranks of this disk's slots compare alike for any */
                    int64_t rk, rx;
                    const Leaf L = event_ranks(C, lane, S, my.paul, Sh.ctr, rk, rx);
                    double kA, kB;
                    halves(L.key, kA, kB);
                    double lim = min_f64(kA, kB);
                    if (Wc.ls > 0) {
                        int xA, xB;
                        halves(L.aux, xA, xB);
                        const int64_t rA = lane_value64(L.rank, 0), rB = lane_value64(L.rank, 32);
                        double limA, limB;
                        path_nodes(A, lane, Wc.ls, P, p, kA, xA, rA, pj, kB, xB, rB,
                                   Sh.nodes[wave], limA, limB);
                        lim = min_f64(lim, limA);
                        /* the partner's own event, which this one takes away,
                         * hid the rest of its group */
                        if (pj >= 0 && Wc.idx[pj >> (6 * Wc.ls)] == pj)
                            lim = min_f64(lim, limB);
                    }
                    const bool coll = S.kind == EVK_COLLISION, wall = W && S.kind == EVK_WALL;
                    int flags = (coll ? WS_COLL : 0) | (wall ? WS_WALL : 0);
                    if (__ballot(S.ov)) flags |= WS_OV;
                    halves(S.cx | (S.cy << 16), cellA, cellB);
                    if (S.kind == EVK_CROSSING) {
                        S.n1 -= S.cy * C.ncx + S.cx == S.c0 ? 1 : 0;
                        if (S.n1 >= C.cap) flags |= WS_FULL;
                        const int oy = S.c0 / C.ncx;
                        cellB = (S.c0 - oy * C.ncx) | (oy << 16);
                    }
                    const int type = aux >= 0 ? EDMD_EV_COLLISION : (wall ? EDMD_EV_WALL : EDMD_EV_CELLCROSS);
                    brief = WB_INS * event_inserts(S);
                    if (type == EDMD_EV_CELLCROSS) brief |= WB_CROSS;
                    if ((flags & (WS_OV | WS_FULL)) || !(t <= ra.tmax) || (ra.stop_mask & (1 << type)))
                        brief |= WB_LAST;
                    if (coll || wall) brief |= WB_COUNTED;
                    if (C.tape_cap > 0 && !G && (coll || (wall && S.d != 2))) brief |= WB_TAPED;
                    pj2 = pj;
                    WideSlot& me = Sh.slot[wave];
                    if (lane == 0) {
                        me.key = t;
                        me.lim = lim;
                        if (wall) {
                            me.dp[0] = S.dp;
                            me.dp[1] = S.dpl;
                            me.dp[2] = S.dpm;
                            me.dp[3] = S.dpr;
                        }
                        me.p = p;
                        me.j = pj >= 0 ? pj : -2;
                        me.ca = cellA;
                        me.cb = cellB;
                        me.flags = flags;
                        me.type = type;
                        me.gp = p >> (6 * Wc.ls);
                        me.gj = pj >= 0 ? pj >> (6 * Wc.ls) : -2;
                    }
                }
                lds_barrier();

                /* check: lane k tests the event of wavefront k < this one's */
                if (my.plain) {
                    const int reach = (W && !G && (C.field_on || C.damping)) ? 2 : 1;
                    const int k = lane < wave ? lane : 0;
                    const WideSlot& o = Sh.slot[k];
                    const WidePick& ok = Sh.pick[k];
                    const int p = my.p, q = my.aux >= 0 ? my.aux : -1;
                    const int op = o.p, oj = o.j;
                    const bool same = (p == op) | (p == oj) | (q == op) | (q == oj);
                    const bool near = cells_near(cellA, o.ca, reach, C.ncx, C.ncy) ||
                                      cells_near(cellA, o.cb, reach, C.ncx, C.ncy) ||
                                      cells_near(cellB, o.ca, reach, C.ncx, C.ncy) ||
                                      cells_near(cellB, o.cb, reach, C.ncx, C.ncy);
                    const bool zero = S.none0 && (op == 0 || oj == 0);
                    /* a stale event takes nothing away */
                    const bool back = !(o.flags & WS_COLL) && my.ord > ok.shad;
                    const bool late = !(my.key < o.lim);
                    /* several leaves of one window node: it is made from memory */
                    const int gp = p >> (6 * Wc.ls), gj = pj2 >= 0 ? pj2 >> (6 * Wc.ls) : -3;
                    const bool share = (gp == o.gp) | (gp == o.gj) | (gj == o.gp) | (gj == o.gj);
                    const bool on = lane < wave && ok.plain != 0;
                    if (!__ballot(on && (same || near || zero || back || late))) brief |= WB_OK;
                    if (Wc.ls > 0 && __ballot(on && share)) brief |= WB_SHARE;
                }
                if (lane == 0) Sh.verdict[wave] = brief;
                lds_barrier();

                /* commit */
                const WideVerdict V = wide_verdict<NW>(Sh, lane);
                const int cut = wide_cut<NW>(V, __builtin_amdgcn_readfirstlane(Sh.room),
                                             __builtin_amdgcn_readfirstlane(Sh.croom));
                const bool share = Wc.ls > 0 && (V.share & ((1u << cut) - 1)) != 0;
                if (tid == 0) {
                    Sh.cut = cut;
                    Sh.sums = cut;
                    Sh.lim = Sh.pick[cut - 1].key + Sh.state.width;
                }
                if (wave < cut) {
                    const double t = my.key;
                    const int p = my.p, aux = my.aux;
                    const int64_t trace = Sh.ntrace + wave;
                    int64_t rk, rx;
                    const Leaf L = event_ranks(C, lane, S, my.paul, Sh.ctr + wide_inserts(V, wave), rk, rx);
                    if (C.trace_cap > 0 && lane == 0 && trace < C.trace_cap) {
                        EdmdTraceRec rec;
                        rec.type = Sh.slot[wave].type;
                        rec.i = p;
                        rec.j = aux >= 0 ? aux : S.d;
                        rec.valid = S.kind != EVK_STALE;
                        rec.t = t;
                        A.trace[trace] = rec;
                    }
                    if (S.kind == EVK_CROSSING) event_cells(C, A, lane, S);
                    if (!(S.kind == EVK_CROSSING && S.n1 >= C.cap)) {
                        event_store(A, lane, t, S);
                        if (W && !G && (C.field_on || C.damping)) {
                            WAVE_SYNC();
                            fly_neighbours(C, A, lane, t, S, Sh.cand[wave]);
                        }
                        if (S.kind == EVK_CROSSING) event_enter(C, A, lane, S, S.n1);
                        if (!G && (brief & WB_TAPED) && lane == 0) {
                            if (S.kind == EVK_COLLISION) {
                                const WideSlot& me = Sh.slot[wave];
                                S.dx = me.ax;
                                S.dy = me.ay;
                                S.dvx = me.cx;
                                S.dvy = me.cy;
                                S.ff = me.ff;
                            }
                            tape_store<W>(C, A, t, S, p, aux,
                                          Sh.ntape + __popc(V.taped & ((1u << wave) - 1)));
                        }
                        event_slots(A, lane, S, L, rk, rx);
                        if (Wc.ls == 0) {
                            if ((lane & 31) == 0 && (lane == 0 || S.nown == 2)) {
                                Wc.key[S.own] = L.key;
                                Wc.rank[S.own] = L.rank;
                                Wc.aux[S.own] = L.aux;
                            }
                        } else if (!share) {
                            const int64_t rA = lane_value64(L.rank, 0), rB = lane_value64(L.rank, 32);
                            if (lane == 0) nodes_store(A, Wc, p, rA, S.nown == 2 ? aux : -1, rB, Sh.nodes[wave]);
                        }
                    }
                }
                if (Wc.ls > 0 && share) {
                    __syncthreads();
                    for (int l = 1; l <= Wc.ls; ++l) {
                        if (wave < cut) {
                            node_make(C, A, Wc, lane, l, my.p, my.key);
                            if (S.nown == 2) node_make(C, A, Wc, lane, l, my.aux, my.key);
                        }
                        if (l < Wc.ls) __syncthreads();
                    }
                }
                lds_barrier();
            }
        }
        const EdmdConst& C = opaque(Cs);
        const AR& A = opaque(As);
        if (todo == WT_STOP) break;
        if (tid == 0 && todo == WT_SPECIAL) {
            WideState& Z = Sh.state;
            Z.R.t = Z.R.next_special;
            Z.R.nevents++;
            Z.last_type = Z.R.special;
            Z.guard = 0;
            if (C.trace_cap > 0) {
                if (Z.ntrace < C.trace_cap) {
                    EdmdTraceRec rec;
                    rec.type = Z.R.special;
                    rec.i = 0;
                    rec.j = 0;
                    rec.valid = 1;
                    rec.t = Z.R.t;
                    A.trace[Z.ntrace] = rec;
                }
                ++Z.ntrace;
            }
        }
        __syncthreads();
        LoopRegs H = Sh.state.R; /* on every wavefront */
        const int sp = H.special;
        __syncthreads();
        bool ov = false;
        if (todo == WT_WRAP) {
            /* the overflow list filed again (refile_wrap's steps) */
            wide_refile<NT>(C, A, tid, H.paul, H.win, H.ctr, &Sh.moved, &Sh.ctr);
            if (Sh.moved) cal_build<NT>(C, A, Wc, tid);
        } else if (sp == EDMD_EV_SCREENSHOT) {
            ev_screenshot<NT, G, W>(C, A, tid, H);
        } else if (sp == EDMD_EV_THERMO) {
            ev_thermo<NT>(C, A, tid, H, Sh.vir, Sh.red);
        } else {
            if (sp == EDMD_EV_GROWSTOP) ov = G && ev_stop_grow<NT, W>(C, A, tid, H, Sh.red);
            else ov = ev_rescale<NT, G, W>(C, A, tid, H, Sh.red);
            ov = __syncthreads_or(ov ? 1 : 0) != 0;
            cal_build<NT>(C, A, Wc, tid);
        }
        __syncthreads();
        if (wave == 0) {
            WideState Z = Sh.state;
            LoopRegs& R = Z.R;
            R.ctr = H.ctr;
            if (todo == WT_SPECIAL) {
                if (ov && R.status == EDMD_DEV_OK) {
                    R.status = EDMD_DEV_OVERLAP;
                    if (sp == EDMD_EV_GROWSTOP) R.err_i = 0;
                }
                if (G && sp == EDMD_EV_GROWSTOP) {
                    R.ncol = 0; /* stopGrow resets ncol and ncross, EDMD.c:4745-4746 */
                    Z.ncross = 0;
                    Z.reason = EDMD_STOP_GROWN;
                } else if (ra.stop_mask & (1 << sp)) {
                    Z.reason = EDMD_STOP_SPECIAL;
                }
            }
            next_special(A.st, R);
            if (lane == 0) {
                Sh.state = Z;
                Sh.cut = 0;
                Sh.lim = R.t + Z.width;
                Sh.lcount = 0;
            }
        }
        __syncthreads();
        if (todo == WT_SPECIAL &&
            ((G && sp == EDMD_EV_GROWSTOP) || (ra.stop_mask & (1 << sp))))
            break;
    }
    __syncthreads();
    const EdmdConst& C = opaque(Cs);
    const AR& A = opaque(As);
    if (tid == 0) {
        EdmdState* st = A.st;
        const WideState& Z = Sh.state;
        const LoopRegs& R = Z.R;
        st->t = R.t;
        st->ncol = R.ncol;
        st->ncross = Z.ncross;
        st->nevents = R.nevents;
        st->status = R.status;
        st->err_i = R.err_i;
        st->err_j = R.err_j;
        st->stop_reason = Z.reason;
        st->last_type = Z.last_type;
        st->paul = R.paul;
        st->ctr = R.ctr;
        st->win = R.win;
        st->ntape = Z.ntape;
        st->ntrace = Z.ntrace;
        for (int k = 0; k < 4; ++k) st->vir[k] = Sh.vir[k];
    }
    cal_close<NT>(C, A, Wc, tid);
}

/* The arrays in HBM, the calendar's window level in the dynamic LDS.  FLAT:
 * the window is of leaves for every system, so none of the code for the
 * levels between, whose path of nodes took 30 registers: 128 of them and 16
 * wavefronts a CU, where one kernel for both held 239 and 8 (one system of
 * 2000 disks, 4000 collisions: 6.20 ms to 4.84 with 16 wavefronts). */
template <int NW, bool FLAT, bool G, bool W>
__global__ __launch_bounds__(64 * NW, (FLAT || NW > 8) ? 4 : 2) void k_wide(
    const EdmdSys* __restrict__ systems, EdmdRunArgs ra) {
    extern __shared__ __align__(64) unsigned char lds_pool[];
    const EdmdSys& S = systems[blockIdx.x];
    if ((uni(S.a.st->growing) != 0) != G) return;
    wide_loop<NW, FLAT, G, W>(S.c, S.a, ra, (unsigned char EDMD_LDS*)lds_pool);
}

/* The arrays in LDS as well (edmd_lds.h). */
template <int NW, bool G, bool W>
__global__ __launch_bounds__(64 * NW, 4) void k_wide_lds(const EdmdSys* __restrict__ systems,
                                                         EdmdRunArgs ra) {
    extern __shared__ __align__(64) unsigned char lds_pool[];
    const EdmdSys& S = systems[blockIdx.x];
    if ((uni(S.a.st->growing) != 0) != G) return;
    __shared__ EdmdArraysL A;
    unsigned char EDMD_LDS* base = (unsigned char EDMD_LDS*)lds_pool;
    const uint32_t used = lds_carve<G>(S.c, S.a, base, A);
    __syncthreads();
    lds_system<true, G, 64 * NW>(S.c, S.a, A, threadIdx.x);
    __syncthreads();
    wide_loop<NW, true, G, W>(S.c, A, ra, base + used);
    __syncthreads();
    lds_system<false, G, 64 * NW>(S.c, S.a, A, threadIdx.x);
}

template <int NW, bool G, bool W>
const void* kernel_of(int place) {
    if (place == EDMD_WIDE_LDS) return (const void*)k_wide_lds<NW, G, W>;
    if (place == EDMD_WIDE_LEAVES) return (const void*)k_wide<NW, true, G, W>;
    return (const void*)k_wide<NW, false, G, W>;
}

} // namespace

template <bool G, bool W>
const void* EdmdWideVariant<G, W>::kernel(int waves, int place) {
    if (waves == 16) return kernel_of<16, G, W>(place);
    if (waves == 8) return kernel_of<8, G, W>(place);
    if (waves == 4) return kernel_of<4, G, W>(place);
    return nullptr;
}

template <bool G, bool W>
hipError_t EdmdWideVariant<G, W>::run(int waves, int place, const EdmdSys* d_sys, int nsys,
                                      size_t dyn_bytes, EdmdRunArgs ra, hipStream_t s) {
    const void* f = kernel(waves, place);
    if (!f) return hipErrorInvalidValue;
    ra.nsys = nsys;
    void* args[] = {(void*)&d_sys, (void*)&ra};
    return hipLaunchKernel(f, dim3(nsys), dim3(64 * waves), args, dyn_bytes, s);
}

template struct EdmdWideVariant<EDMD_LOOP_GROW, EDMD_LOOP_WALLS>;
