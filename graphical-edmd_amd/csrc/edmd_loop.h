/*
 * The event loop's device code: the emulated queue position, the handlers
 * of scheduled and particle events and the loop itself, templates over the
 * arrays' residency (HBM or LDS), the calendar depth, growth and walls.
 * Reference line numbers are those of src/EDMD.c.
 */
#ifndef EDMD_LOOP_H
#define EDMD_LOOP_H

#include "edmd_event.h"

/* ------------------------------------------------------------ event loop */

/* Loop state kept in registers; the rest of EdmdState stays in memory and
 * is touched only by the events that use it. */
/* The emulated state of the reference's queue, kept in LDS (one wavefront
 * per workgroup): it changes rarely and would otherwise hold scalar
 * registers through the whole loop. */
struct QueueState {
    int32_t cand[EDMD_STAGE_MAX]; /* candidate stage of the neighbour scan */
    /* the top level of the calendar (at most 64 nodes): read by every
     * event, written only here while the loop runs and copied to HBM when
     * it ends */
    EdmdNode top[64];
    /* collision virial sums since the last thermo row (collTermX, collTermY,
     * collTermXY, collTermYX), accumulated by lane 0 in the reference's
     * order; here rather than in scalar registers, which the loop has too
     * few of */
    double vir[4];
    /* the calendar's minimum after a wrap moved particle events of the
     * overflow list (moved != 0) */
    double mkey;
    int32_t mleaf, maux, moved;
    /* the loop's registers between its inner loop and a scheduled event */
    double t, paul;
    int64_t ctr, win;
    uint64_t ncol, nevents, ncross;
    int32_t status, err_i, err_j, last_type;
};

/* Top level of the calendar between HBM and the LDS copy. */
template <class AR>
__device__ __forceinline__ void top_load(const EdmdConst& C, const AR& A, int lane,
                                         EdmdNode* top) {
    if (lane < C.lsize[C.nlev]) top[lane] = level(A, C.nlev)[lane];
    WAVE_SYNC();
}

template <class AR>
__device__ __forceinline__ void top_store(const EdmdConst& C, const AR& A, int lane,
                                          const EdmdNode* top) {
    if (lane < C.lsize[C.nlev]) level(A, C.nlev)[lane] = top[lane];
    WAVE_SYNC();
}

struct LoopRegs {
    double t;
    double next_special; /* earliest of the screenshot / thermo / noise / growth-stop times */
    int special;         /* its kind */
    uint64_t ncol, nevents;
    int32_t status, err_i, err_j;
    /* the queue's position (uniform, kept in scalar registers) */
    double paul;   /* the reference's paulTime */
    int64_t ctr;   /* insertions so far */
    int64_t win;   /* buckets passed */
    int64_t srank; /* rank of the next special event */
    int64_t swin;  /* bucket of the next special event (-1: overflow list) */
    int cur;       /* win modulo the bucket count */
    QueueState* q; /* LDS: candidate stage and the calendar's top level */
};

__device__ __forceinline__ void next_special(const EdmdState* st, LoopRegs& R) {
    double tsp = st->next_screen;
    int64_t rsp = st->rank_screen, wsp = st->win_screen;
    int sp = EDMD_EV_SCREENSHOT;
    if (before(st->next_thermo, st->rank_thermo, tsp, rsp)) {
        tsp = st->next_thermo; rsp = st->rank_thermo; wsp = st->win_thermo; sp = EDMD_EV_THERMO;
    }
    if (before(st->next_noise, st->rank_noise, tsp, rsp)) {
        tsp = st->next_noise; rsp = st->rank_noise; wsp = st->win_noise; sp = EDMD_EV_ADDINGNOISE;
    }
    if (before(st->next_grow, st->rank_grow, tsp, rsp)) {
        tsp = st->next_grow; rsp = st->rank_grow; wsp = st->win_grow; sp = EDMD_EV_GROWSTOP;
    }
    R.next_special = uni(tsp);
    R.srank = uni64(rsp);
    R.swin = uni64(wsp);
    R.special = uni(sp);
}

/* Bucket the reference files an event at t_ev into (addEventToQueue,
 * EDMD.c:2144-2170): the current one when t_ev - paulTime < dtPaul, -1 for
 * the overflow list, else win + (int)((t_ev - paulTime) / dtPaul). */
__device__ __host__ __forceinline__ int64_t window_of(double t_ev, double paul, double dtp,
                                                      int nlists, int64_t win) {
    const double dt = t_ev - paul;
    if (dt < dtp) return win;
    if (dt >= dtp * nlists) return -1;
    return win + (int64_t)(int)(dt / dtp);
}

/* The overflow list's special events filed again when the ring of buckets
 * wraps (EDMD.c:2292-2302): they get their bucket and rank anew. */
__device__ __forceinline__ void refile_specials(const EdmdConst& C, EdmdState* st, double paul,
                                             int64_t win, int64_t& ctr) {
    double* ts[4] = {&st->next_screen, &st->next_thermo, &st->next_noise, &st->next_grow};
    int64_t* ws[4] = {&st->win_screen, &st->win_thermo, &st->win_noise, &st->win_grow};
    int64_t* rs[4] = {&st->rank_screen, &st->rank_thermo, &st->rank_noise, &st->rank_grow};
    for (int k = 0; k < 4; ++k) {
        const double tk = *ts[k];
        if (*ws[k] != -1 || !(tk < 1e25)) continue;
        const int64_t w = window_of(tk, paul, C.dtp, C.nlists, win);
        /* filed straight into the tree during the wrap, before the new
         * bucket is drained: ahead of both drained and later direct events */
        const int64_t r = (w == win) ? ctr : rank_of(tk, paul, C.dtp, C.horizon, ctr);
        ctr++;
        WAVE_SYNC();
        if ((threadIdx.x & 63) == 0) {
            *ws[k] = w;
            *rs[k] = r;
        }
        WAVE_SYNC();
    }
}

/* Rank of a particle event of the overflow list filed again at a wrap with
 * counter c (addEventToQueue from addNextPaulEvent, EDMD.c:2144-2170,
 * 2292-2302): straight into the tree, which is empty during a wrap, so
 * ahead of the drained bucket and of every later insertion (rank c, as a
 * special filed there); the overflow list again; or a bucket. */
__device__ __forceinline__ int64_t refiled_rank(const EdmdConst& C, double t_ev, double paul,
                                                int64_t c) {
    const double dt = t_ev - paul;
    if (dt < C.dtp) return c;
    if (dt >= C.horizon) return EDMD_RANK_OVF + c;
    return EDMD_RANK_DIRECT - 1 - c;
}

/* The slots of disk k that wait in the overflow list, filed again at a wrap
 * of the bucket ring with the counter at now: a slot ranked EDMD_RANK_OVF + c
 * gets the counter 2 now - 1 - c.  Returns whether its leaf was made again. */
template <class AR>
__device__ __forceinline__ bool refile_disk(const EdmdConst& C, const AR& A, int k, double paul,
                                            int64_t now) {
    int64_t rk = A.erank[2 * k], rx = A.erank[2 * k + 1];
    const bool fk = EDMD_RANK_IS_OVF(rk), fx = EDMD_RANK_IS_OVF(rx);
    if (!fk && !fx) return false;
    const EdmdEv e = A.e[k];
    if (fk) rk = refiled_rank(C, e.tcoll, paul, 2 * now - 1 - (rk - EDMD_RANK_OVF));
    if (fx) rx = refiled_rank(C, e.tcross, paul, 2 * now - 1 - (rx - EDMD_RANK_OVF));
    A.erank[2 * k] = rk;
    A.erank[2 * k + 1] = rx;
    const Leaf Lf = make_leaf(e.tcoll, rk, e.tcross, rx, e.partner, e.dir);
    EdmdNode nd;
    nd.key = Lf.key;
    nd.idx = k;
    nd.aux = Lf.aux;
    A.leaf[k] = nd;
    A.lrank[k] = Lf.rank;
    return true;
}

/* The particle events of the overflow list filed again at a wrap
 * (EDMD.c:2292-2302), after its special events, in the order of the list's
 * walk from its head (the newest first): a slot ranked EDMD_RANK_OVF + c
 * gets the counter 2 now - 1 - c and the rank of where it goes now; the
 * counter moves past them all (the list holds counters from the previous
 * wrap's on).  The leaves of the disks concerned are made again and the
 * calendar is rebuilt.  Once per wrap of the bucket ring (5 time units);
 * run from the loop's body, like the thermostat, not from the bucket walk,
 * which stays small. */
template <class AR>
__device__ void rebuild_tree(const EdmdConst& C, const AR& A, int lane);

/* The overflow list filed again at a wrap (EDMD.c:2292-2302): its special
 * events, then its particle events in the order of the list's walk from
 * its head (the newest first): a slot ranked EDMD_RANK_OVF + c gets the
 * counter 2 now - 1 - c and the rank of where it goes now, and the counter
 * moves past them all (the list holds counters from the previous wrap's
 * on).  When any slot moved, the leaves of the disks concerned are made
 * again, the calendar is rebuilt, its top level reloaded and its minimum
 * left in q (q->moved = 1).  Once per wrap of the bucket ring (5 time
 * units); kept out of line, with the loop's registers out of its way. */
template <class AR>
__device__ __noinline__ void refile_wrap(const EdmdConst& C, const AR& A, QueueState* q,
                                         double paul, int64_t win, double t, int64_t& ctr) {
    const int lane = threadIdx.x & 63;
    refile_specials(C, A.st, paul, win, ctr);
    const int64_t now = ctr;
    bool any = false;
    for (int k = lane; k < C.n; k += 64) any |= refile_disk(C, A, k, paul, now);
    const bool moved = __ballot(any) != 0ull;
    const int64_t lo = A.st->ovf_lo;
    WAVE_SYNC();
    if (lane == 0) A.st->ovf_lo = now;
    ctr = 2 * now - lo;
    if (moved) {
        WAVE_SYNC();
        rebuild_tree(C, A, lane);
        top_load(C, A, lane, q->top);
        double key;
        int leaf, aux;
        top_min(C, A, lane, q->top, t, key, leaf, aux);
        if (lane == 0) {
            q->mkey = key;
            q->mleaf = leaf;
            q->maux = aux;
        }
    }
    if (lane == 0) q->moved = moved ? 1 : 0;
    WAVE_SYNC();
}

/* One bucket further (addNextPaulEvent, EDMD.c:2287-2307); true when the
 * ring wrapped (the overflow list filed again, refile_wrap). */
template <class AR>
__device__ __forceinline__ bool step_window(const EdmdConst& C, const AR& A, LoopRegs& R) {
    R.paul = uni(R.paul + C.dtp);
    R.win++;
    if (++R.cur < C.nlists) return false;
    R.cur = 0;
    int64_t ctr = R.ctr;
    refile_wrap(C, A, R.q, R.paul, R.win, R.t, ctr);
    R.ctr = uni64(ctr);
    return true;
}

/* findNextEvent (EDMD.c:2313-2327): while no pending event is in the
 * reference's tree -- a particle event within dtPaul of paulTime, or a
 * special event whose bucket has come up -- move on one bucket (refiling
 * the overflow list when the ring wraps).  Then the earlier in the tree by
 * (time, rank) is next.  Returns true for the special event, false for
 * the particle event (key, leaf, aux: the calendar's minimum, taken anew
 * when a wrap moved particle events of the overflow list).  A queue whose next event lies
 * more than 2^24 buckets ahead is not walked bucket by bucket (the
 * reference would); paulTime then jumps to that event. */
template <class AR>
__device__ __forceinline__ bool pick_next(const EdmdConst& C, const AR& A, EdmdState* st,
                                          LoopRegs& R, double& key, int& leaf, int& aux) {
    /* the particle event's rank matters only against a special at its time */
    auto krank = [&]() { return key == R.next_special ? uni64(A.lrank[leaf]) : (int64_t)0; };
    for (int guard = 0;; ++guard) {
        const bool part_in = key - R.paul < C.dtp;
        const int64_t ws = R.swin;
        const bool spec_in = ws >= 0 && ws <= R.win;
        if (part_in || spec_in)
            return spec_in && (!part_in || before(R.next_special, R.srank, key, krank()));
        if (!(key < 1e25) && !(R.next_special < 1e25)) return R.next_special <= key;
        if (guard >= (1 << 24)) {
            const double tn = key < R.next_special ? key : R.next_special;
            while (!(tn - R.paul < C.dtp)) {
                R.paul = uni(R.paul + C.dtp);
                R.win++;
            }
            return before(R.next_special, R.srank, key, krank());
        }
        if (step_window(C, A, R)) {
            next_special(st, R);
            if (R.q->moved) {
                key = R.q->mkey;
                leaf = R.q->mleaf;
                aux = R.q->maux;
            }
        }
    }
}

/* Rank of the next insertion; counts it. */
__device__ __forceinline__ int64_t take_rank(const EdmdConst& C, LoopRegs& R, double t_ev) {
    const int64_t r = rank_of(t_ev, R.paul, C.dtp, C.horizon, R.ctr);
    R.ctr++;
    return r;
}

template <class AR>
__device__ __forceinline__ void trace_push(const EdmdConst& C, const AR& A, int lane,
                                           double t, int type, int i, int j, int valid) {
    if (C.trace_cap <= 0) return;
    if (lane == 0) {
        const int64_t k = A.st->ntrace;
        if (k < C.trace_cap) {
            EdmdTraceRec rec;
            rec.type = type;
            rec.i = i;
            rec.j = j;
            rec.valid = valid;
            rec.t = t;
            A.trace[k] = rec;
        }
        A.st->ntrace = k + 1;
    }
}

/* A group of NT threads runs the handlers of scheduled events: one wavefront
 * (the serial loop) or the whole workgroup (the wide loop). */
template <int NT>
__device__ __forceinline__ void group_sync() {
    if (NT > 64) __syncthreads();
    else WAVE_SYNC();
}

/* Ordered sum over all particles of f(q), accumulated in particle order as
 * the reference's serial loops do (physicalQ, EDMD.c:5968-6013).  The first
 * wavefront adds; the chain of additions is the bound (n times the latency
 * of one), so each value comes by readlane, not by an LDS shuffle per
 * addition, and the next 64 values are read ahead.  red: LDS through which
 * a group of several wavefronts gets the sum. */
template <int NT, class F>
__device__ __forceinline__ double ordered_sum(int n, int tid, double* red, F f) {
    double acc = 0;
    if (NT == 64 || tid < 64) {
        const int lane = tid & 63;
        double next = lane < n ? f(lane) : 0.0;
        int base = 0;
        for (; base + 64 <= n; base += 64) {
            const double v = next;
            const int q = base + 64 + lane;
            next = q < n ? f(q) : 0.0;
#pragma unroll
            for (int l = 0; l < 64; ++l) acc += lane_value(v, l);
        }
        for (int l = 0; l < n - base; ++l) acc += lane_value(next, l);
        if (NT > 64 && lane == 0) red[0] = acc;
    }
    if (NT > 64) {
        __syncthreads();
        acc = red[0];
        __syncthreads();
    }
    return acc;
}

template <int NT, bool G, bool W, class AR>
__device__ __forceinline__ void ev_screenshot(const EdmdConst& C, const AR& A, int tid,
                                              LoopRegs& R) {
    /* takeAScreenshot, EDMD.c:4657-4677: free-fly every particle */
    const double t = R.t;
    for (int q = tid; q < C.n; q += NT) {
        const auto r = A.p + q;
        double x = r->x, y = r->y, tl = r->tl;
        if (G) {
            double rad = r->rad;
            fly_grow(C, t, x, y, r->vx, r->vy, tl, rad, A.vr[q]);
            r->rad = rad;
        } else {
            double vx = r->vx, vy = r->vy;
            fly_v<W>(C, t, x, y, vx, vy, tl);
            if (W) {
                r->vx = vx;
                r->vy = vy;
            }
        }
        r->x = x;
        r->y = y;
        r->tl = tl;
    }
    group_sync<NT>();
    const int64_t wk = window_of(t + C.dtime, R.paul, C.dtp, C.nlists, R.win);
    const int64_t rk = take_rank(C, R, t + C.dtime);
    if (tid == 0) {
        A.st->next_screen = t + C.dtime;
        A.st->rank_screen = rk;
        A.st->win_screen = wk;
    }
    group_sync<NT>();
}

template <int NT, class AR>
__device__ __forceinline__ void ev_thermo(const EdmdConst& C, const AR& A, int tid, LoopRegs& R,
                                          double* vir, double* red) {
    /* takeAThermo + saveThermo, EDMD.c:4679-4713, 5232-5333 */
    const double t = R.t;
    const uint64_t ncol = R.ncol;
    const int64_t wk = window_of(t + C.dtime_thermo, R.paul, C.dtp, C.nlists, R.win);
    const int64_t rk = take_rank(C, R, t + C.dtime_thermo);
    const auto P = A.p;
    double E = ordered_sum<NT>(C.n, tid, red, [&](int q) {
        double a = P[q].vx;
        return 0.5 * P[q].m * (a * a + P[q].vy * P[q].vy);
    });
    double ex = ordered_sum<NT>(C.n, tid, red, [&](int q) { return P[q].m * P[q].vx * P[q].vx; });
    double ey = ordered_sum<NT>(C.n, tid, red, [&](int q) { return P[q].m * P[q].vy * P[q].vy; });
    double exy = ordered_sum<NT>(C.n, tid, red, [&](int q) { return P[q].m * P[q].vx * P[q].vy; });
    double eyx = ordered_sum<NT>(C.n, tid, red, [&](int q) { return P[q].m * P[q].vy * P[q].vx; });
    /* the mid wall's columns (EDMD.c:5453-5477), from the stored disks in
     * particle order; type-0 disks on the other side add +0 */
    double nl = 0, nr = 0, ns = 0, tl = 0, tr = 0, tsol = 0;
    if (C.walls & 8) {
        const auto T = A.ptype;
        const double h = C.halfLx;
        auto temp = [&](int q) {
            return 0.5 * P[q].m * (P[q].vx * P[q].vx + P[q].vy * P[q].vy);
        };
        nl = ordered_sum<NT>(C.n, tid, red, [&](int q) { return (T[q] == 0 && P[q].x < h) ? 1.0 : 0.0; });
        nr = ordered_sum<NT>(C.n, tid, red, [&](int q) { return (T[q] == 0 && P[q].x > h) ? 1.0 : 0.0; });
        ns = ordered_sum<NT>(C.n, tid, red, [&](int q) { return T[q] != 0 ? 1.0 : 0.0; });
        tl = ordered_sum<NT>(C.n, tid, red, [&](int q) { return (T[q] == 0 && P[q].x < h) ? temp(q) : 0.0; });
        tr = ordered_sum<NT>(C.n, tid, red, [&](int q) { return (T[q] == 0 && P[q].x > h) ? temp(q) : 0.0; });
        tsol = ordered_sum<NT>(C.n, tid, red, [&](int q) { return T[q] != 0 ? temp(q) : 0.0; });
    }
    EdmdState* st = A.st;
    /* EDMD.c:5253-5256: the disc's area inside a circular wall */
    const double area = (C.walls & 4) ? 3.14159265358979323846 * C.halfLx * C.halfLx : C.Lx * C.Ly;
    const double dT = t - st->last_thermo;
    const double v0 = vir[0], v1 = vir[1], v2 = vir[2], v3 = vir[3];
    const int k = st->nthermo;
    if (tid == 0) {
        if (k < C.thermo_cap) {
            EdmdThermoRow row;
            row.t = t;
            row.ncol = ncol;
            row.e_per_n = E / C.n;
            row.pxx = -1 * v0 / (area * dT) + ex / area;
            row.pyy = -1 * v1 / (area * dT) + ey / area;
            row.pxy = -1 * v2 / (area * dT) + exy / area;
            row.pyx = -1 * v3 / (area * dT) + eyx / area;
            row.pressure = (-1 / (dT)) * (v0 + v1) / (2 * area) + E / area;
            row.pwall = 0;
            row.pmid = row.dp_lr = row.pack_left = row.pack_right = 0;
            row.temp_left = row.temp_right = row.temp_solute = 0;
            if (C.walls & 8) {
                const double ratio = 3.14159265358979323846 / (C.halfLx * C.Ly);
                const double sr = C.sizeratio;
                row.pmid = st->dpm / (dT * C.Ly);
                row.dp_lr = -(st->dpr - st->dpl) / (dT * C.Ly);
                row.pack_left = ratio * (double)(int)nl * sr * sr;
                row.pack_right = ratio * (double)(int)nr * sr * sr;
                row.temp_left = tl / (int)nl;
                row.temp_right = tr / (int)nr;
                row.temp_solute = tsol / (int)ns;
            }
            if (C.walls & 7) {
                /* EDMD.c:5428-5451: dp / (deltaTime * perimeter) */
                double perimeter = 0;
                if (C.walls & 4) perimeter = 3.14159265358979323846 * C.Lx;
                if (C.walls & 1) perimeter += 2 * C.Ly;
                if (C.walls & 2) perimeter += 2 * C.Lx;
                row.pwall = st->dpw / (dT * perimeter);
            }
            A.thermo[k] = row;
        }
        if (C.walls & 7) st->dpw = 0;
        if (C.walls & 8) st->dpl = st->dpm = st->dpr = 0;
        st->nthermo = k + 1;
        st->last_thermo = t;
        st->next_thermo = t + C.dtime_thermo;
        st->rank_thermo = rk;
        st->win_thermo = wk;
    }
    if (tid == 0) vir[0] = vir[1] = vir[2] = vir[3] = 0;
    group_sync<NT>();
}

template <int NT, bool G, bool W, class AR>
__device__ __forceinline__ bool ev_rescale(const EdmdConst& C, const AR& A, int tid,
                                           LoopRegs& R, double* red) {
    const double t = R.t;
    /* addNoise, velocity-rescale branch (noise == 2): EDMD.c:4828-4832,
     * 4880-4915, 4922 */
    const auto P = A.p;
    double E = ordered_sum<NT>(C.n, tid, red, [&](int q) {
        double a = P[q].vx;
        return 0.5 * P[q].m * (a * a + P[q].vy * P[q].vy);
    });
    for (int q = tid; q < C.n; q += NT) {
        EdmdPart r = A.p[q];
        r.coll = r.coll + 1;
        if (G) fly_grow(C, t, r.x, r.y, r.vx, r.vy, r.tl, r.rad, A.vr[q]);
        else fly_v<W>(C, t, r.x, r.y, r.vx, r.vy, r.tl);
        r.vx /= sqrt(E / C.n / C.temperature);
        r.vy /= sqrt(E / C.n / C.temperature);
        A.p[q] = r;
    }
    group_sync<NT>();
    bool ov = false;
    /* per particle: crossing, then collision (EDMD.c:4909-4915) */
    for (int q = tid; q < C.n; q += NT)
        ov |= sweep_one<G, W>(C, A, t, q, R.paul, R.ctr + 2 * (int64_t)q, R.ctr + 2 * (int64_t)q + 1);
    R.ctr += 2 * (int64_t)C.n;
    const bool any_ov = __ballot(ov) != 0ull;
    group_sync<NT>();
    const int64_t wk = window_of(t + C.dtnoise, R.paul, C.dtp, C.nlists, R.win);
    const int64_t rk = take_rank(C, R, t + C.dtnoise);
    if (tid == 0) {
        A.st->next_noise = t + C.dtnoise;
        A.st->rank_noise = rk;
        A.st->win_noise = wk;
    }
    group_sync<NT>();
    return any_ov;
}

__device__ __forceinline__ void flag_overlap(LoopRegs& R, bool ov, int p) {
    if (__ballot(ov) != 0ull && R.status == EDMD_DEV_OK) {
        R.status = EDMD_DEV_OVERLAP;
        R.err_i = p;
    }
}

/* stopGrow, EDMD.c:4740-4785 (2D, no wells): final flight with growth, all
 * counters and image counters reset, normalizePhysicalQ (EDMD.c:5723-5764:
 * remove the mean momentum, scale to E/N = Einit), then the Normal
 * prediction of every disk with stopGrow's partner counters, and a new
 * calendar.  The caller continues in the Normal loop. */
template <int NT, bool W, class AR>
__device__ __forceinline__ bool ev_stop_grow(const EdmdConst& C, const AR& A, int tid,
                                             LoopRegs& R, double* red) {
    const double t = R.t;
    for (int q = tid; q < C.n; q += NT) {
        EdmdPart r = A.p[q];
        fly_grow(C, t, r.x, r.y, r.vx, r.vy, r.tl, r.rad, A.vr[q]);
        r.coll = 0;
        A.p[q] = r;
        A.img[2 * q] = 0;
        A.img[2 * q + 1] = 0;
    }
    group_sync<NT>();
    const auto P = A.p;
    const int n = C.n;
    if (!(W && (C.walls & 4))) {
        const double px = ordered_sum<NT>(n, tid, red, [&](int q) { return P[q].vx * P[q].m; });
        const double py = ordered_sum<NT>(n, tid, red, [&](int q) { return P[q].vy * P[q].m; });
        for (int q = tid; q < n; q += NT) {
            const double m = P[q].m;
            P[q].vx -= px / (n * m);
            P[q].vy -= py / (n * m);
        }
    } else {
        /* in a circle, the angular momentum about the centre
         * (EDMD.c:5730-5749): dvT accumulates -m (x0 vy - y0 vx), dvM m r */
        const double h = C.halfLx;
        const double dvT = -ordered_sum<NT>(n, tid, red, [&](int q) {
            return P[q].m * (-P[q].vx * (P[q].y - h) + P[q].vy * (P[q].x - h));
        });
        const double dvM = ordered_sum<NT>(n, tid, red, [&](int q) {
            return P[q].m * sqrt((P[q].x - h) * (P[q].x - h) + (P[q].y - h) * (P[q].y - h));
        });
        const double dv = dvT / dvM;
        for (int q = tid; q < n; q += NT) {
            const double x0 = P[q].x - h, y0 = P[q].y - h;
            const double r = sqrt(x0 * x0 + y0 * y0);
            P[q].vx += -dv * y0 / r;
            P[q].vy += dv * x0 / r;
        }
    }
    group_sync<NT>();
    const double E = ordered_sum<NT>(n, tid, red, [&](int q) {
        double a = P[q].vx;
        return 0.5 * P[q].m * (a * a + P[q].vy * P[q].vy);
    });
    for (int q = tid; q < n; q += NT) {
        P[q].vx /= sqrt(E / n / C.einit);
        P[q].vy /= sqrt(E / n / C.einit);
        P[q].coll = 1;
    }
    group_sync<NT>();
    bool ov = false;
    /* per particle: collision, then crossing (EDMD.c:4770-4776) */
    for (int q = tid; q < n; q += NT)
        ov |= sweep_one<false, W>(C, A, t, q, R.paul, R.ctr + 2 * (int64_t)q + 1,
                               R.ctr + 2 * (int64_t)q, true);
    R.ctr += 2 * (int64_t)n;
    group_sync<NT>();
    const bool any_ov = __ballot(ov) != 0ull;
    if (tid == 0) {
        A.st->growing = 0;
        A.st->next_grow = INF_D;
    }
    group_sync<NT>();
    return any_ov;
}

/* Rebuilds every level of the calendar after a full re-prediction. */
template <class AR>
__device__ void rebuild_tree(const EdmdConst& C, const AR& A, int lane) {
    for (int l = 1; l <= C.nlev; ++l) {
        for (int g = lane; g < C.lsize[l]; g += 64) node_min(C, A, l, g);
        WAVE_SYNC();
    }
}

/* A particle event of the serial loop (doTheCollisionNormal / Grow,
 * EDMD.c:3465-3915, doTheCrossing, EDMD.c:2501-2590, doTheWallNormal / Grow,
 * EDMD.c:3333-3460): p's leaf holds the current time and code aux.  Returns
 * the kind of event handled (EDMD_EV_*). */
template <int ML, bool G, bool W, class AR>
__device__ __forceinline__ int ev_particle(const EdmdConst& C, const AR& A, int lane, LoopRegs& R,
                                           int p, int aux) {
    /* what follows from the lane alone is made again for each event, not
     * held in registers through the loop */
    asm volatile("" : "+v"(lane));
    PathCache<ML> P;
    path_prefetch<ML>(C, A, lane, p, aux >= 0 ? aux : -1, P);
    const double t = R.t;
    EvState S;
    event_open<G, W>(C, A, lane, t, p, aux, S);
    const bool wall = W && S.kind == EVK_WALL;
    trace_push(C, A, lane, t,
               aux >= 0 ? EDMD_EV_COLLISION : (wall ? EDMD_EV_WALL : EDMD_EV_CELLCROSS), p,
               aux >= 0 ? aux : S.d, S.kind != EVK_STALE);
    if (S.kind == EVK_COLLISION || wall) R.ncol++;
    if (S.kind == EVK_CROSSING) {
        /* into a full cell: the disk's record stays as it was */
        event_cells(C, A, lane, S);
        const int c1 = S.cy * C.ncx + S.cx;
        const int n1 = A.ccnt[c1];
        if (n1 >= C.cap) {
            if (R.status == EDMD_DEV_OK) {
                R.status = EDMD_DEV_CELL_OVERFLOW;
                R.err_i = p;
                R.err_j = c1;
            }
            return EDMD_EV_CELLCROSS;
        }
        event_store(A, lane, t, S);
        event_enter(C, A, lane, S, n1);
    } else {
        event_store(A, lane, t, S);
        if (S.kind != EVK_STALE) event_sums<G, W>(C, A, lane, t, S, p, aux, R.q->vir);
    }
    WAVE_SYNC();
    event_predict<G, W, false>(C, A, lane, t, S, R.q->cand);
    flag_overlap(R, S.ov, p);
    int64_t rk, rx;
    const Leaf L = event_ranks(C, lane, S, R.paul, R.ctr, rk, rx);
    R.ctr += event_inserts(S);
    event_slots(A, lane, S, L, rk, rx);
    const double kA = lane_value(L.key, 0), kB = lane_value(L.key, 32);
    const int xA = __builtin_amdgcn_readlane(L.aux, 0), xB = __builtin_amdgcn_readlane(L.aux, 32);
    path_update<ML>(C, A, lane, P, p, kA, xA, S.nown == 2 ? aux : -1, kB, xB, R.q->top, t);
    return aux >= 0 ? EDMD_EV_COLLISION : (wall ? EDMD_EV_WALL : EDMD_EV_CELLCROSS);
}

/* A reference the compiler cannot look through: what it loads through one
 * is not kept in registers past the next.  The system's record does not
 * change during a launch: constant memory, read with scalar loads. */
template <class T>
__device__ __forceinline__ const T& opaque_const(const T& r) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef const T __attribute__((address_space(4))) * ConstPtr;
    ConstPtr p = (ConstPtr)&r;
    asm volatile("" : "+s"(p));
    return *(const T*)p;
#else
    return r;
#endif
}
__device__ __forceinline__ const EdmdConst& opaque(const EdmdConst& r) { return opaque_const(r); }
__device__ __forceinline__ const EdmdArrays& opaque(const EdmdArrays& r) { return opaque_const(r); }
template <class AR>
__device__ __forceinline__ const AR& opaque(const AR& r) { return r; }

/* A scheduled event (screenshot, thermo row, rescale, growth stop), the
 * loop's registers handed over through its LDS state. */
template <bool G, bool W, class AR>
__device__ __forceinline__ void special_event(const EdmdConst& C, const AR& A, int lane,
                                              QueueState* q, int sp) {
    LoopRegs R;
    R.q = q;
    R.t = q->t;
    R.paul = q->paul;
    R.ctr = uni64(q->ctr);
    R.win = uni64(q->win);
    R.ncol = q->ncol;
    bool ov = false;
    if (sp == EDMD_EV_SCREENSHOT) {
        ev_screenshot<64, G, W>(C, A, lane, R);
    } else if (sp == EDMD_EV_THERMO) {
        ev_thermo<64>(C, A, lane, R, q->vir, nullptr);
    } else {
        if (sp == EDMD_EV_GROWSTOP) ov = G && ev_stop_grow<64, W>(C, A, lane, R, nullptr);
        else ov = ev_rescale<64, G, W>(C, A, lane, R, nullptr);
        rebuild_tree(C, A, lane);
        top_load(C, A, lane, q->top);
    }
    WAVE_SYNC();
    if (lane == 0) {
        q->ctr = R.ctr;
        if (ov && q->status == EDMD_DEV_OK) {
            q->status = EDMD_DEV_OVERLAP;
            if (sp == EDMD_EV_GROWSTOP) q->err_i = 0;
        }
        if (G && sp == EDMD_EV_GROWSTOP) {
            q->ncol = 0; /* stopGrow resets ncol and ncross, EDMD.c:4745-4746 */
            q->ncross = 0;
        }
    }
    WAVE_SYNC();
}

/* Persistent event loop of one system on one wavefront; ML bounds the
 * calendar depth of every system in the launch.  A holds the system's arrays
 * in HBM (EdmdArrays) or in LDS (EdmdArraysL); the caller has checked that
 * the system's growth phase matches G.
 *
 * Particle events run in an inner loop of their own; a scheduled event
 * leaves it, with the loop's registers and the system's record let go (the
 * record is read again through an opaque reference), so that the scheduled
 * events' sweeps and sums cost the inner loop no registers: with them in the
 * same loop it spilled 61-106 scalar registers into vector ones. */
template <int ML, bool G, bool W, int WPB = 1, class AR>
__device__ __forceinline__ void run_loop(const EdmdConst& Cs, const AR& As, EdmdRunArgs ra) {
    /* WPB wavefronts per workgroup, each looping over its own system with
     * its own LDS queue state */
    const int lane = threadIdx.x & 63;
    __shared__ QueueState Qs[WPB];
    QueueState* const q = &Qs[WPB > 1 ? wave_in_group() : 0];
    int reason = EDMD_STOP_NONE;
    {
        const EdmdState* st = As.st;
        if (lane == 0) {
            q->t = st->t;
            q->paul = st->paul;
            q->ctr = st->ctr;
            q->win = st->win;
            q->ncol = st->ncol;
            q->nevents = st->nevents;
            q->ncross = st->ncross;
            q->status = st->status;
            q->err_i = st->err_i;
            q->err_j = st->err_j;
            q->last_type = st->last_type;
            for (int k = 0; k < 4; ++k) q->vir[k] = st->vir[k];
        }
        top_load(Cs, As, lane, q->top);
    }
    WAVE_SYNC();
    for (;;) {
        int sp = -1;
        {
            const EdmdConst& C = opaque(Cs);
            const AR& A = opaque(As);
            EdmdState* st = A.st;
            LoopRegs R;
            R.q = q;
            R.t = q->t;
            R.ncol = q->ncol;
            R.nevents = q->nevents;
            R.status = q->status;
            R.err_i = q->err_i;
            R.err_j = q->err_j;
            R.paul = q->paul;
            R.ctr = uni64(q->ctr);
            R.win = uni64(q->win);
            R.cur = (int)(R.win % C.nlists);
            uint64_t ncross = q->ncross;
            int last_type = q->last_type;
            next_special(st, R);
            const int64_t ev_limit = st->ev_limit < ra.max_events ? st->ev_limit : ra.max_events;
            const uint64_t coll_limit = st->coll_limit < ra.max_coll ? st->coll_limit : ra.max_coll;
            for (;;) {
                if (R.status != EDMD_DEV_OK) { reason = EDMD_STOP_ERROR; break; }
                if ((int64_t)R.nevents >= ev_limit) { reason = EDMD_STOP_EVENTS; break; }
                if (R.ncol >= coll_limit) { reason = EDMD_STOP_COLLISIONS; break; }
                if (!(R.t <= ra.tmax)) { reason = EDMD_STOP_TIME; break; }
                double key;
                int p, aux;
                top_min(C, A, lane, R.q->top, R.t, key, p, aux);
                if (!(key < INF_D) && !(R.next_special < INF_D)) { reason = EDMD_STOP_EMPTY; break; }
                if (pick_next(C, A, st, R, key, p, aux)) {
                    sp = R.special;
                    R.t = R.next_special;
                    trace_push(C, A, lane, R.t, sp, 0, 0, 1);
                    R.nevents++;
                    last_type = sp;
                    break;
                }
                R.t = key;
                last_type = ev_particle<ML, G, W>(C, A, lane, R, p, aux);
                if (last_type == EDMD_EV_CELLCROSS) ncross++;
                R.nevents++;
                if (ra.stop_mask & (1 << last_type)) { reason = EDMD_STOP_SPECIAL; break; }
            }
            WAVE_SYNC();
            if (lane == 0) {
                q->t = R.t;
                q->ncol = R.ncol;
                q->nevents = R.nevents;
                q->ncross = ncross;
                q->status = R.status;
                q->err_i = R.err_i;
                q->err_j = R.err_j;
                q->paul = R.paul;
                q->ctr = R.ctr;
                q->win = R.win;
                q->last_type = last_type;
            }
            WAVE_SYNC();
        }
        if (sp < 0) break;
        special_event<G, W>(opaque(Cs), opaque(As), lane, q, sp);
        if (G && sp == EDMD_EV_GROWSTOP) { reason = EDMD_STOP_GROWN; break; }
        if (ra.stop_mask & (1 << sp)) { reason = EDMD_STOP_SPECIAL; break; }
    }
    const AR& A = opaque(As);
    if (lane == 0) {
        EdmdState* st = A.st;
        st->t = q->t;
        st->ncol = q->ncol;
        st->ncross = q->ncross;
        st->nevents = q->nevents;
        st->status = q->status;
        st->err_i = q->err_i;
        st->err_j = q->err_j;
        st->stop_reason = reason;
        st->last_type = q->last_type;
        st->paul = q->paul;
        st->ctr = q->ctr;
        st->win = q->win;
        for (int k = 0; k < 4; ++k) st->vir[k] = q->vir[k];
    }
    top_store(opaque(Cs), A, lane, q->top);
}

#endif
