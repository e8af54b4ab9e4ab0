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
 *            gathered from LDS
 *   leader   the first wavefront orders them, leaves out those that an
 *            earlier one takes away (a collision re-predicts its partner,
 *            whose own event, often the same collision seen from the other
 *            disk, then never pops) and gives wavefront w the w-th of the rest
 *   compute  every wavefront works out its event without writing
 *            (event_open, event_predict<SPEC>)
 *   check    every wavefront tests its event against the ones before it: it
 *            must be earlier than anything they predict and read no disk or
 *            cell that they write
 *   commit   the longest prefix that the serial loop would handle in the same
 *            way (no failed test, no scheduled event, ring wrap or bound in
 *            it) is written: insertion counters, sums, tape and trace
 *            positions follow from the events' order in it
 * The first event of a round always commits, so the loop advances whatever
 * the limit or the spatial distribution; scheduled events and ring wraps are
 * handled between rounds by the whole workgroup.  The ordering is the first
 * wavefront's alone: done by all eight alike it took twice as long, two
 * wavefronts sharing each SIMD's issue.
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
constexpr int WIDE_LIST = 32; /* entries an order takes */

/* An event as the leader hands it to a wavefront. */
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
    double dp[4];    /* its momentum to the walls */
};

enum { WS_COLL = 1, WS_WALL = 2, WS_OV = 4, WS_FULL = 8 };

/* A wavefront's byte of the round's verdict. */
enum { WB_OK = 1, WB_LAST = 2, WB_COUNTED = 4, WB_TAPED = 8, WB_INS = 16, WB_SHARE = 128 };
constexpr uint64_t WB_EACH = 0x0101010101010101ull;

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
    int32_t solo; /* the next round handles the earliest event alone */
    int32_t halt; /* a kind of event that stops the run was handled */
};

template <int NW>
struct WideShared {
    int32_t cand[NW][EDMD_STAGE_MAX];
    WideState state;
    WidePick pick[NW];
    WideSlot slot[NW];
    PathNodes nodes[NW];
    WideEntry list[WIDE_LIST];
    int32_t shad[WIDE_LIST];
    uint64_t verdict; /* a byte per wavefront */
    int32_t lcount, todo, cut, sums, moved; /* cut: events the last round committed */
    int32_t room, croom; /* events and counted events that the bounds leave */
    double lim;          /* the scan's time limit */
    double vir[4];
    double red[2];
    int64_t ctr, ntape, ntrace;
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
        const bool tie = ((at >> lane) & 1) != 0;
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

/* The leader's part of a round: orders the gathered nodes, leaves out what an
 * earlier one takes away and fills the picks; the buckets up to each event
 * (pick_next) are counted in plain steps, an event behind a ring wrap or a
 * scheduled event is not plain.  Returns WT_ROUND, or what must happen before
 * the earliest event. */
template <int NW, bool W, class AR>
__device__ __forceinline__ int wide_order(const EdmdConst& C, const AR& A, int lane,
                                          const WideCal& Wc, WideShared<NW>& Sh) {
    WideState& Z = Sh.state;
    LoopRegs& R = Z.R;
    double width = Z.width;
    int n = Sh.lcount;
    if (n < 1 || n > WIDE_LIST) {
        if (Z.tries < 12) {
            /* no usable window: another limit */
            ++Z.tries;
            width *= n > WIDE_LIST ? 0.5 : 4.0;
            if (!(width > 0)) width = 1e-300;
            Z.width = width;
            if (lane == 0) {
                Sh.lcount = 0;
                Sh.lim = R.t + width;
            }
            return WT_SCAN;
        }
        n = -1;
    }
    /* the next window: about two events a wavefront */
    if (n >= 0 && n < NW + NW / 2) width = width * 1.2 + 1e-300;
    else if (n > 2 * NW + NW / 4) width = width * 0.85;
    Z.width = width;
    double key;
    int p, aux;
    bool shadowed = false, stop = false;
    if (n > 0) {
        /* lanes e and 32 + e: entry e of the list, against every other one
         * (even ones on the lower half, odd ones on the upper): its place by
         * (time, rank), and the one whose partner it is */
        const int e = lane & 31, h = lane >> 5;
        const bool in = e < n;
        const WideEntry me = Sh.list[in ? e : 0];
        p = me.p;
        int place = 0, by = -1, count = 0;
        for (int i = 0; i < n; i += 8) {
            WideEntry o[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) o[c] = Sh.list[(i + 2 * c + h) & (WIDE_LIST - 1)];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int k = i + 2 * c + h;
                const bool real = k < n;
                const bool sooner = (o[c].key < me.key) | ((o[c].key == me.key) & (o[c].rank < me.rank));
                const bool hit = real & (o[c].aux == p);
                place += (real & sooner) ? 1 : 0;
                by = hit ? k : by;
                count += hit ? 1 : 0;
            }
        }
        int u, v;
        halves(place, u, v);
        place = in ? u + v : e;
        halves(by, u, v);
        by = u > v ? u : v;
        halves(count, u, v);
        count = u + v;
        /* taken away by entry `by`, if that comes earlier; where it is itself
         * taken away, or several name this disk, the window ends here */
        const int bat = 4 * (by < 0 ? 0 : by);
        const int bplace = __builtin_amdgcn_ds_bpermute(bat, place);
        shadowed = in && by >= 0 && bplace < place;
        const int bshadowed = __builtin_amdgcn_ds_bpermute(bat, shadowed ? 1 : 0);
        stop = in && by >= 0 && ((count > 1 && place > 0) || (shadowed && bshadowed));
        /* by place, on lanes 0 .. n - 1 */
        const int from = 4 * (__builtin_amdgcn_ds_permute(4 * place, lane) & 31);
        const int flag = (shadowed ? 1 : 0) | (stop ? 2 : 0) | (bplace << 2);
        const int sflag = __builtin_amdgcn_ds_bpermute(from, flag);
        const long long kb = __double_as_longlong(me.key);
        const int klo = __builtin_amdgcn_ds_bpermute(from, (int)kb);
        const int khi = __builtin_amdgcn_ds_bpermute(from, (int)(kb >> 32));
        key = __longlong_as_double(((long long)khi << 32) | (unsigned int)klo);
        p = __builtin_amdgcn_ds_bpermute(from, p);
        aux = __builtin_amdgcn_ds_bpermute(from, me.aux);
        shadowed = (sflag & 1) != 0;
        stop = (sflag & 2) != 0 && lane < n;
        if (lane < WIDE_LIST) Sh.shad[lane] = 64;
        WAVE_SYNC();
        if (lane < n && shadowed) atomicMin(&Sh.shad[sflag >> 2], lane);
        WAVE_SYNC();
    } else {
        /* many equal times, or none pending: the earliest event alone */
        key = INF_D;
        int64_t rank = 0;
        int node = 0;
        for (int g = lane; g < Wc.m; g += 64) {
            const double k = Wc.key[g];
            if (k < key || (k == key && k < INF_D && Wc.rank[g] < rank)) {
                key = k;
                rank = Wc.rank[g];
                node = g;
            }
        }
        int leaf = Wc.ls > 0 ? Wc.idx[node] : node, who = lane;
        double kk = key;
        wave_argmin(A, R.t, kk, leaf, who);
        key = kk;
        node = __builtin_amdgcn_readlane(node, who);
        p = Wc.ls > 0 ? Wc.idx[node] : node;
        aux = Wc.aux[node];
        n = 1;
        if (lane < WIDE_LIST) Sh.shad[lane] = 64;
        WAVE_SYNC();
    }
    Z.tries = 0;
    const double k0 = lane_value(key, 0);
    const int p0 = __builtin_amdgcn_readlane(p, 0);
    if (lane == 0) {
        Sh.lcount = 0;
        Sh.lim = k0 + width; /* of the next scan, unless the time moves on */
    }
    if (!(k0 < INF_D) && !(R.next_special < INF_D)) return WT_STOP;
    /* the buckets up to each event */
    uint64_t use = __ballot(lane < n && !shadowed);
    const uint64_t end = __ballot(stop);
    if (end) use &= ((uint64_t)1 << __builtin_ctzll(end)) - 1;
    if (Z.solo) use = 1;
    const int pos = (int)__popcll(use & (((uint64_t)1 << lane) - 1));
    const bool mine = ((use >> lane) & 1) != 0 && pos < NW;
    double paul = R.paul;
    int steps = 0;
    bool plain = mine && key < INF_D && key < R.next_special && !(R.swin >= 0 && R.swin <= R.win);
    while (plain && !(key - paul < C.dtp)) {
        paul = paul + C.dtp;
        ++steps;
        if (R.cur + steps >= C.nlists || steps > 4096 || (R.swin >= 0 && R.swin <= R.win + steps))
            plain = false;
    }
    if (W && C.thermal_wall && pos > 0 && aux <= EDMD_WALL_CODE(0)) plain = false;
    if (Z.solo && lane == 0) {
        plain = true;
        paul = R.paul;
        steps = 0;
    }
    if (__ballot(lane == 0 && plain) == 0) {
        /* the earliest event is not a plain one: findNextEvent's decision
         * (EDMD.c:2313-2327), one ring wrap at a time */
        for (;; ++Z.guard) {
            const bool part_in = k0 - R.paul < C.dtp;
            const bool spec_in = R.swin >= 0 && R.swin <= R.win;
            auto sooner = [&]() {
                return before(R.next_special, R.srank, k0,
                              k0 == R.next_special ? uni64(A.lrank[p0]) : (int64_t)0);
            };
            bool special;
            if (part_in || spec_in) {
                special = spec_in && (!part_in || sooner());
            } else if (!(k0 < 1e25) && !(R.next_special < 1e25)) {
                special = R.next_special <= k0;
            } else if (Z.guard >= (1 << 24)) {
                const double tn = k0 < R.next_special ? k0 : R.next_special;
                while (!(tn - R.paul < C.dtp)) {
                    R.paul = R.paul + C.dtp;
                    R.win++;
                }
                special = sooner();
            } else {
                R.paul = R.paul + C.dtp;
                R.win++;
                if (++R.cur >= C.nlists) {
                    R.cur = 0;
                    ++Z.guard;
                    return WT_WRAP;
                }
                continue;
            }
            if (special) return WT_SPECIAL;
            /* a particle event after all: alone in a round of its own */
            Z.solo = 1;
            if (lane == 0) Sh.lim = k0 + width;
            return WT_SCAN;
        }
    }
    if (lane < NW) Sh.pick[lane].plain = 0;
    WAVE_SYNC();
    if (mine) {
        WidePick& k = Sh.pick[pos];
        k.key = key;
        k.paul = paul;
        k.p = p;
        k.aux = aux;
        k.steps = steps;
        k.plain = plain ? 1 : 0;
        k.ord = lane;
        k.shad = Sh.shad[lane & (WIDE_LIST - 1)];
    }
    return WT_ROUND;
}

/* The events of a round that commit, from its verdict: up to the first one
 * that failed its test, the first after which the loop stops, the bounds. */
template <int NW>
__device__ __forceinline__ int wide_cut(uint64_t verdict, int room, int croom) {
    const uint64_t all = NW == 8 ? ~(uint64_t)0 : ((uint64_t)1 << (8 * (NW & 7))) - 1;
    const uint64_t fail = ~verdict & WB_EACH & all, last = (verdict >> 1) & WB_EACH;
    int cut = NW;
    if (fail) cut = (int)__builtin_ctzll(fail) >> 3;
    if (last) {
        const int c = ((int)__builtin_ctzll(last) >> 3) + 1;
        cut = c < cut ? c : cut;
    }
    cut = room < cut ? room : cut;
    if (croom <= NW) {
        int c = 0, m = 0;
        for (; m < cut && c < croom; ++m) c += (int)(verdict >> (8 * m + 2)) & 1;
        cut = m;
    }
    return cut;
}

/* The verdict's bytes below wavefront m. */
__device__ __forceinline__ uint64_t wide_below(uint64_t verdict, int m) {
    return m >= 8 ? verdict : verdict & (((uint64_t)1 << (8 * m)) - 1);
}

__device__ __forceinline__ int wide_inserts(uint64_t v) {
    return (int)(__popcll((v >> 4) & WB_EACH) + 2 * __popcll((v >> 5) & WB_EACH) +
                 4 * __popcll((v >> 6) & WB_EACH));
}

/* The loop's state after a round of `cut` events (the leader's first lane),
 * and what the next round needs of it. */
template <int NW>
__device__ __forceinline__ void wide_advance(const EdmdConst& C, WideShared<NW>& Sh, int cut,
                                             int stop_mask, int64_t ev_limit, uint64_t coll_limit) {
    WideState& Z = Sh.state;
    LoopRegs& R = Z.R;
    if (cut == 0) {
        /* no round since the state was read or a scheduled event */
        const int64_t er = ev_limit - (int64_t)R.nevents;
        const uint64_t cr = coll_limit - R.ncol;
        Sh.room = er < NW ? (int)er : NW;
        Sh.croom = cr <= NW ? (int)cr : NW + 1;
        Sh.ctr = R.ctr;
        Sh.ntape = Z.ntape;
        Sh.ntrace = Z.ntrace;
        return;
    }
    const uint64_t done = wide_below(Sh.verdict, cut);
    const WideSlot& last = Sh.slot[cut - 1];
    const WidePick& lp = Sh.pick[cut - 1];
    const int type = last.type, flags = last.flags, nins = wide_inserts(done);
    int ncr = 0;
#pragma unroll
    for (int m = 0; m < NW; ++m) ncr += (m < cut && Sh.slot[m].type == EDMD_EV_CELLCROSS) ? 1 : 0;
    const double t = lp.key;
    int64_t ctr = R.ctr + nins;
    R.t = t;
    R.paul = lp.paul;
    R.win += lp.steps;
    R.cur += lp.steps;
    R.ncol += __popcll((done >> 2) & WB_EACH);
    R.nevents += cut;
    Z.last_type = type;
    if (C.trace_cap > 0) Z.ntrace += cut;
    Z.ntape += __popcll((done >> 3) & WB_EACH);
    Z.ncross += ncr;
    Z.guard = 0;
    Z.solo = 0;
    if (stop_mask & (1 << type)) Z.halt = 1;
    if (flags & WS_FULL) {
        R.status = EDMD_DEV_CELL_OVERFLOW;
        R.err_i = last.p;
        R.err_j = (last.ca >> 16) * C.ncx + (last.ca & 0xffff);
        ctr -= 2; /* the crossing stops before its insertions */
    } else if (flags & WS_OV) {
        R.status = EDMD_DEV_OVERLAP;
        R.err_i = last.p;
    }
    R.ctr = ctr;
    /* for the round that follows */
    const int64_t er = ev_limit - (int64_t)R.nevents;
    const uint64_t cr = coll_limit - R.ncol;
    Sh.room = er < NW ? (int)er : NW;
    Sh.croom = cr <= NW ? (int)cr : NW + 1;
    Sh.ctr = ctr;
    Sh.ntape = Z.ntape;
    Sh.ntrace = Z.ntrace;
}

template <int NW, bool G, bool W, class AR>
__device__ __forceinline__ void wide_loop(const EdmdConst& Cs, const AR& As, EdmdRunArgs ra,
                                          unsigned char EDMD_LDS* pool) {
    constexpr int NT = 64 * NW;
    static_assert(NW <= 8, "a byte of the verdict per wavefront");
    __shared__ WideShared<NW> Sh;
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_group();
    WideCal Wc;
    {
        const EdmdConst& C = opaque(Cs);
        const AR& A = opaque(As);
        const EdmdState* st = A.st;
        Wc.ls = edmd_wide_level(&C);
        Wc.m = C.lsize[Wc.ls];
        Wc.key = (double EDMD_LDS*)pool;
        Wc.rank = (int64_t EDMD_LDS*)(pool + (size_t)Wc.m * 8);
        Wc.aux = (int32_t EDMD_LDS*)(pool + (size_t)Wc.m * 16);
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
        Z.guard = Z.tries = Z.solo = Z.halt = 0;
        Z.reason = EDMD_STOP_NONE;
        if (tid < 4) Sh.vir[tid] = st->vir[tid];
        if (tid == 0) {
            Sh.state = Z;
            Sh.cut = 0;
            Sh.lcount = 0;
            Sh.sums = 0;
            Sh.verdict = 0;
            Sh.lim = R.t + Z.width;
        }
        cal_build<NT>(C, A, Wc, tid);
    }
    for (;;) {
        int todo;
        {
            const EdmdConst& C = opaque(Cs);
            const AR& A = opaque(As);
            EdmdState* st = A.st;
            const int64_t ev_limit = st->ev_limit < ra.max_events ? st->ev_limit : ra.max_events;
            const uint64_t coll_limit = st->coll_limit < ra.max_coll ? st->coll_limit : ra.max_coll;
            const int reach = (W && !G && (C.field_on || C.damping)) ? 2 : 1;
            for (;;) {
                /* scan (the others), the state after the last round (the
                 * leader's first lane) */
                if (wave == 0) {
                    if (lane == 0)
                        wide_advance<NW>(C, Sh, Sh.cut, ra.stop_mask, ev_limit, coll_limit);
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
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const uint64_t in = __ballot(k[u] < lim);
                            if (!in) continue;
                            int at = 0;
                            if (lane == 0) at = atomicAdd(&Sh.lcount, (int)__popcll(in));
                            at = __builtin_amdgcn_readfirstlane(at) +
                                 (int)__popcll(in & (((uint64_t)1 << lane) - 1));
                            if (k[u] < lim && at < WIDE_LIST) {
                                const int g = g0 + u * (NT - 64);
                                WideEntry e;
                                e.key = k[u];
                                e.rank = Wc.rank[g];
                                e.p = Wc.ls > 0 ? Wc.idx[g] : g;
                                e.aux = Wc.aux[g];
                                Sh.list[at] = e;
                            }
                        }
                    }
                }
                __syncthreads();
                if (wave == 0) {
                    WideState& Z = Sh.state;
                    const LoopRegs& R = Z.R;
                    int td = WT_STOP;
                    if (Z.halt) Z.reason = EDMD_STOP_SPECIAL;
                    else if (R.status != EDMD_DEV_OK) Z.reason = EDMD_STOP_ERROR;
                    else if ((int64_t)R.nevents >= ev_limit) Z.reason = EDMD_STOP_EVENTS;
                    else if (R.ncol >= coll_limit) Z.reason = EDMD_STOP_COLLISIONS;
                    else if (!(R.t <= ra.tmax)) Z.reason = EDMD_STOP_TIME;
                    else {
                        td = wide_order<NW, W>(C, A, lane, Wc, Sh);
                        if (td == WT_STOP) Z.reason = EDMD_STOP_EMPTY;
                    }
                    if (lane == 0) Sh.todo = td;
                } else if (wave == 1 && !G) {
                    /* the last round's sums, in its events' order */
                    const int cut = Sh.sums;
                    if (lane < 4) {
                        double v = Sh.vir[lane];
                        for (int m = 0; m < cut; ++m) {
                            const double u = Sh.slot[m].vir[lane];
                            if (Sh.slot[m].flags & WS_COLL) v += u;
                        }
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
                lds_barrier();
                todo = Sh.todo;
                if (todo == WT_SCAN) {
                    if (tid == 0) Sh.cut = 0;
                    lds_barrier(); /* read by all before the leader writes it again */
                    continue;
                }
                if (todo != WT_ROUND) break;

                /* compute */
                const WidePick& my = Sh.pick[wave];
                EvState S;
                int brief = 0, cellA = 0, cellB = 0, pj2 = -1;
                if (my.plain) {
                    const double t = my.key;
                    const int p = my.p, aux = my.aux;
                    event_open<G, W>(C, A, lane, t, p, aux, S);
                    PathWindow P;
                    const int pj = S.nown == 2 ? aux : -1;
                    if (Wc.ls > 0) path_window(C, A, lane, Wc.ls, p, pj, P);
                    event_predict<G, W, true>(C, A, lane, t, S, Sh.cand[wave]);
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
                    if ((flags & (WS_OV | WS_FULL)) || !(t <= ra.tmax) || (ra.stop_mask & (1 << type)))
                        brief |= WB_LAST;
                    if (coll || wall) brief |= WB_COUNTED;
                    if (C.tape_cap > 0 && !G && (coll || (wall && S.d != 2))) brief |= WB_TAPED;
                    pj2 = pj;
                    WideSlot& me = Sh.slot[wave];
                    if (coll && !G && lane < 4) {
                        const double u = (lane & 1) == 0 ? S.dx : S.dy;
                        const double v = (lane == 0 || lane == 3) ? S.dx : S.dy;
                        me.vir[lane] = S.w * u * v;
                    }
                    if (lane == 0) {
                        me.key = t;
                        me.lim = lim;
                        if (coll && !G && C.tape_cap > 0)
                            me.wsum = S.w * (S.dx * S.dx + S.dy * S.dy);
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
                    const bool late = !(my.key > ok.key && my.key < o.lim);
                    /* several leaves of one window node: it is made from memory */
                    const int gp = p >> (6 * Wc.ls), gj = pj2 >= 0 ? pj2 >> (6 * Wc.ls) : -3;
                    const bool share = (gp == o.gp) | (gp == o.gj) | (gj == o.gp) | (gj == o.gj);
                    const bool on = lane < wave && ok.plain != 0;
                    if (!__ballot(on && (same || near || zero || back || late))) brief |= WB_OK;
                    if (Wc.ls > 0 && __ballot(on && share)) brief |= WB_SHARE;
                }
                if (lane == 0) ((unsigned char*)&Sh.verdict)[wave] = (unsigned char)brief;
                lds_barrier();

                /* commit */
                const uint64_t verdict = (uint64_t)uni64((int64_t)Sh.verdict);
                const int cut = wide_cut<NW>(verdict, __builtin_amdgcn_readfirstlane(Sh.room),
                                             __builtin_amdgcn_readfirstlane(Sh.croom));
                const uint64_t done = wide_below(verdict, cut);
                const bool share = Wc.ls > 0 && ((done >> 7) & WB_EACH) != 0;
                if (tid == 0) {
                    Sh.cut = cut;
                    Sh.sums = cut;
                    Sh.lim = Sh.pick[cut - 1].key + Sh.state.width;
                }
                if (wave < cut) {
                    const double t = my.key;
                    const int p = my.p, aux = my.aux;
                    const uint64_t prior = wide_below(done, wave);
                    const int64_t trace = Sh.ntrace + wave;
                    int64_t rk, rx;
                    const Leaf L = event_ranks(C, lane, S, my.paul, Sh.ctr + wide_inserts(prior), rk, rx);
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
                        if (!G && (brief & WB_TAPED) && lane == 0)
                            tape_store<W>(C, A, t, S, p, aux,
                                          Sh.ntape + __popcll((prior >> 3) & WB_EACH));
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

/* LDS = false: the system's arrays in HBM, the calendar's window level in
 * the dynamic LDS; LDS = true: the arrays in LDS as well (edmd_lds.h).  Two
 * wavefronts a SIMD: one workgroup of eight, or two of four; without the bound
 * the compiler gave four wavefronts every register, and one CU held one
 * workgroup (512 systems of 400 disks, 4000 collisions each: 18 ms in the loop
 * of one wavefront that ran instead, 12.3 ms here). */
template <int NW, bool G, bool W>
__global__ __launch_bounds__(64 * NW, 2) void k_wide(const EdmdSys* __restrict__ systems,
                                                     EdmdRunArgs ra) {
    extern __shared__ __align__(64) unsigned char lds_pool[];
    const EdmdSys& S = systems[blockIdx.x];
    if ((uni(S.a.st->growing) != 0) != G) return;
    wide_loop<NW, G, W>(S.c, S.a, ra, (unsigned char EDMD_LDS*)lds_pool);
}

template <int NW, bool G, bool W>
__global__ __launch_bounds__(64 * NW, 2) void k_wide_lds(const EdmdSys* __restrict__ systems,
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
    wide_loop<NW, G, W>(S.c, A, ra, base + used);
    __syncthreads();
    lds_system<false, G, 64 * NW>(S.c, S.a, A, threadIdx.x);
}

} // namespace

template <bool G, bool W>
const void* EdmdWideVariant<G, W>::kernel(int waves, int lds) {
    if (waves == 8) return lds ? (const void*)k_wide_lds<8, G, W> : (const void*)k_wide<8, G, W>;
    if (waves == 4) return lds ? (const void*)k_wide_lds<4, G, W> : (const void*)k_wide<4, G, W>;
    return nullptr;
}

template <bool G, bool W>
hipError_t EdmdWideVariant<G, W>::run(int waves, int lds, const EdmdSys* d_sys, int nsys,
                                      size_t dyn_bytes, EdmdRunArgs ra, hipStream_t s) {
    const void* f = kernel(waves, lds);
    if (!f) return hipErrorInvalidValue;
    ra.nsys = nsys;
    void* args[] = {(void*)&d_sys, (void*)&ra};
    return hipLaunchKernel(f, dim3(nsys), dim3(64 * waves), args, dyn_bytes, s);
}

template struct EdmdWideVariant<EDMD_LOOP_GROW, EDMD_LOOP_WALLS>;
