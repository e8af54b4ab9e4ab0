/*
 * The event loop's device code: the emulated queue position, the handlers
 * of scheduled and particle events and the loop itself, templates over the
 * arrays' residency (HBM or LDS), the calendar depth, growth and walls.
 * Reference line numbers are those of src/EDMD.c.
 */
#ifndef EDMD_LOOP_H
#define EDMD_LOOP_H

#include "edmd_device.h"

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
    for (int k = lane; k < C.n; k += 64) {
        int64_t rk = A.erank[2 * k], rx = A.erank[2 * k + 1];
        const bool fk = EDMD_RANK_IS_OVF(rk), fx = EDMD_RANK_IS_OVF(rx);
        if (!fk && !fx) continue;
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
        any = true;
    }
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

/* Ordered sum over all particles of f(q), accumulated in particle order as
 * the reference's serial loops do (physicalQ, EDMD.c:5968-6013). */
template <class F>
__device__ __forceinline__ double ordered_sum(int n, int lane, F f) {
    double acc = 0;
    for (int base = 0; base < n; base += 64) {
        int q = base + lane;
        double v = (q < n) ? f(q) : 0.0;
        int lim = n - base < 64 ? n - base : 64;
        for (int l = 0; l < lim; ++l) {
            double vl = __shfl(v, l, 64);
            acc += vl;
        }
    }
    return acc;
}

template <bool G, bool W, class AR>
__device__ __forceinline__ void ev_screenshot(const EdmdConst& C, const AR& A, int lane,
                                              LoopRegs& R) {
    /* takeAScreenshot, EDMD.c:4657-4677: free-fly every particle */
    const double t = R.t;
    for (int q = lane; q < C.n; q += 64) {
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
    WAVE_SYNC();
    const int64_t wk = window_of(t + C.dtime, R.paul, C.dtp, C.nlists, R.win);
    const int64_t rk = take_rank(C, R, t + C.dtime);
    if (lane == 0) {
        A.st->next_screen = t + C.dtime;
        A.st->rank_screen = rk;
        A.st->win_screen = wk;
    }
    WAVE_SYNC();
}

template <class AR>
__device__ __forceinline__ void ev_thermo(const EdmdConst& C, const AR& A, int lane, LoopRegs& R) {
    /* takeAThermo + saveThermo, EDMD.c:4679-4713, 5232-5333 */
    const double t = R.t;
    const uint64_t ncol = R.ncol;
    const int64_t wk = window_of(t + C.dtime_thermo, R.paul, C.dtp, C.nlists, R.win);
    const int64_t rk = take_rank(C, R, t + C.dtime_thermo);
    const auto P = A.p;
    double E = ordered_sum(C.n, lane, [&](int q) {
        double a = P[q].vx;
        return 0.5 * P[q].m * (a * a + P[q].vy * P[q].vy);
    });
    double ex = ordered_sum(C.n, lane, [&](int q) { return P[q].m * P[q].vx * P[q].vx; });
    double ey = ordered_sum(C.n, lane, [&](int q) { return P[q].m * P[q].vy * P[q].vy; });
    double exy = ordered_sum(C.n, lane, [&](int q) { return P[q].m * P[q].vx * P[q].vy; });
    double eyx = ordered_sum(C.n, lane, [&](int q) { return P[q].m * P[q].vy * P[q].vx; });
    /* the mid wall's columns (EDMD.c:5453-5477), from the stored disks in
     * particle order; type-0 disks on the other side add +0 */
    double nl = 0, nr = 0, ns = 0, tl = 0, tr = 0, tsol = 0;
    if (C.walls & 8) {
        const auto T = A.ptype;
        const double h = C.halfLx;
        auto temp = [&](int q) {
            return 0.5 * P[q].m * (P[q].vx * P[q].vx + P[q].vy * P[q].vy);
        };
        nl = ordered_sum(C.n, lane, [&](int q) { return (T[q] == 0 && P[q].x < h) ? 1.0 : 0.0; });
        nr = ordered_sum(C.n, lane, [&](int q) { return (T[q] == 0 && P[q].x > h) ? 1.0 : 0.0; });
        ns = ordered_sum(C.n, lane, [&](int q) { return T[q] != 0 ? 1.0 : 0.0; });
        tl = ordered_sum(C.n, lane, [&](int q) { return (T[q] == 0 && P[q].x < h) ? temp(q) : 0.0; });
        tr = ordered_sum(C.n, lane, [&](int q) { return (T[q] == 0 && P[q].x > h) ? temp(q) : 0.0; });
        tsol = ordered_sum(C.n, lane, [&](int q) { return T[q] != 0 ? temp(q) : 0.0; });
    }
    EdmdState* st = A.st;
    /* EDMD.c:5253-5256: the disc's area inside a circular wall */
    const double area = (C.walls & 4) ? 3.14159265358979323846 * C.halfLx * C.halfLx : C.Lx * C.Ly;
    const double dT = t - st->last_thermo;
    const double v0 = R.q->vir[0], v1 = R.q->vir[1], v2 = R.q->vir[2], v3 = R.q->vir[3];
    const int k = st->nthermo;
    if (lane == 0) {
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
    if (lane == 0) R.q->vir[0] = R.q->vir[1] = R.q->vir[2] = R.q->vir[3] = 0;
    WAVE_SYNC();
}

/* Rebuilds every level of the calendar after a full re-prediction. */
template <class AR>
__device__ void rebuild_tree(const EdmdConst& C, const AR& A, int lane) {
    for (int l = 1; l <= C.nlev; ++l) {
        for (int g = lane; g < C.lsize[l]; g += 64) node_min(C, A, l, g);
        WAVE_SYNC();
    }
}

template <bool G, bool W, class AR>
__device__ __forceinline__ bool ev_rescale(const EdmdConst& C, const AR& A, int lane,
                                           LoopRegs& R) {
    const double t = R.t;
    /* addNoise, velocity-rescale branch (noise == 2): EDMD.c:4828-4832,
     * 4880-4915, 4922 */
    const auto P = A.p;
    double E = ordered_sum(C.n, lane, [&](int q) {
        double a = P[q].vx;
        return 0.5 * P[q].m * (a * a + P[q].vy * P[q].vy);
    });
    for (int q = lane; q < C.n; q += 64) {
        EdmdPart r = A.p[q];
        r.coll = r.coll + 1;
        if (G) fly_grow(C, t, r.x, r.y, r.vx, r.vy, r.tl, r.rad, A.vr[q]);
        else fly_v<W>(C, t, r.x, r.y, r.vx, r.vy, r.tl);
        r.vx /= sqrt(E / C.n / C.temperature);
        r.vy /= sqrt(E / C.n / C.temperature);
        A.p[q] = r;
    }
    WAVE_SYNC();
    bool ov = false;
    /* per particle: crossing, then collision (EDMD.c:4909-4915) */
    for (int q = lane; q < C.n; q += 64)
        ov |= sweep_one<G, W>(C, A, t, q, R.paul, R.ctr + 2 * (int64_t)q, R.ctr + 2 * (int64_t)q + 1);
    R.ctr += 2 * (int64_t)C.n;
    const bool any_ov = __ballot(ov) != 0ull;
    WAVE_SYNC();
    rebuild_tree(C, A, lane);
    top_load(C, A, lane, R.q->top);
    const int64_t wk = window_of(t + C.dtnoise, R.paul, C.dtp, C.nlists, R.win);
    const int64_t rk = take_rank(C, R, t + C.dtnoise);
    if (lane == 0) {
        A.st->next_noise = t + C.dtnoise;
        A.st->rank_noise = rk;
        A.st->win_noise = wk;
    }
    WAVE_SYNC();
    return any_ov;
}

__device__ __forceinline__ void flag_overlap(LoopRegs& R, bool ov, int p) {
    if (__ballot(ov) != 0ull && R.status == EDMD_DEV_OK) {
        R.status = EDMD_DEV_OVERLAP;
        R.err_i = p;
    }
}

template <int ML, bool W, class AR>
__device__ __forceinline__ void ev_collision(const EdmdConst& C, const AR& A, int lane, LoopRegs& R, int i,
                             int j) {
    /* doTheCollisionNormal, EDMD.c:3542-3562, 3583-3606, 3802-3827, 3869-3879 */
    const EdmdEv ei = A.e[i];
    const int64_t rxi_old = A.erank[2 * i + 1]; /* crossing slot kept by a stale pop */
    const EdmdPart pi = A.p[i];
    const EdmdPart pj = A.p[j];
    PathCache<ML> P;
    path_prefetch<ML>(C, A, lane, i, j, P);
    const double t = R.t;
    double xi = uni(pi.x), yi = uni(pi.y), vxi = uni(pi.vx), vyi = uni(pi.vy), tli = uni(pi.tl);
    const double ri = uni(pi.rad), mi = uni(pi.m);
    const int cxi = uni((int)pi.cx), cyi = uni((int)pi.cy);
    const uint32_t colli = (uint32_t)uni((int)pi.coll);
    const uint32_t collj = (uint32_t)uni((int)pj.coll);
    const uint32_t ca = (uint32_t)uni((int)ei.cact);

    fly_v<W>(C, t, xi, yi, vxi, vyi, tli);
    xi = uni(xi);
    yi = uni(yi);
    vxi = uni(vxi);
    vyi = uni(vyi);
    const bool valid = (ca == collj);
    trace_push(C, A, lane, t, EDMD_EV_COLLISION, i, j, valid ? 1 : 0);
    if (!valid) {
        /* stale prediction: free flight of i and a new collision slot */
        if (lane == 0) {
            A.p[i].x = xi;
            A.p[i].y = yi;
            A.p[i].vx = vxi;
            A.p[i].vy = vyi;
            A.p[i].tl = t;
        }
        WAVE_SYNC();
        const Owner oi{i, xi, yi, vxi, vyi, ri, cxi, cyi};
        bool ov = false;
        double dt, dtb;
        int pa, pb;
        uint32_t cpa, cpb;
        predict_owners<false, W, (ML > 2 && !W)>(C, A, lane, t, 1, oi, oi, dt, pa, cpa, dtb, pb, cpb,
                                                 ov, R.q->cand);
        flag_overlap(R, ov, i);
        const double tk = t + dt;
        const double tci = uni(ei.tcross);
        const int64_t rci = uni64(rxi_old);
        const int diri = uni(ei.dir);
        const int64_t rk = take_rank(C, R, tk);
        if (lane == 0) {
            A.e[i].tcoll = tk;
            A.e[i].partner = pa;
            A.e[i].cact = cpa;
            A.erank[2 * i] = rk;
        }
        path_update<ML>(C, A, lane, P, i, make_leaf(tk, rk, tci, rci, pa, diri), -1, Leaf{}, R.q->top, R.t);
        return;
    }
    R.ncol++;
    double xj = uni(pj.x), yj = uni(pj.y), vxj = uni(pj.vx), vyj = uni(pj.vy), tlj = uni(pj.tl);
    const double rj = uni(pj.rad), mj = uni(pj.m);
    const int cxj = uni((int)pj.cx), cyj = uni((int)pj.cy);
    fly_v<W>(C, t, xj, yj, vxj, vyj, tlj);
    vxj = uni(vxj);
    vyj = uni(vyj);
    double dx = xj - xi;
    double dy = yj - yi;
    double dvx = vxj - vxi;
    double dvy = vyj - vyi;
    double inv_mass = 1 / (mi + mj);
    min_image(C, dx, dy);
    double kernel = inv_mass * (1 + C.res) * (dx * dvx + dy * dvy);
    double ff = kernel / (4 * ri * rj);
    double w = mi * mj * ff;
    vxi = uni(vxi + ff * mj * dx);
    vyi = uni(vyi + ff * mj * dy);
    vxj = uni(vxj - ff * mi * dx);
    vyj = uni(vyj - ff * mi * dy);
    xj = uni(xj);
    yj = uni(yj);
    if (lane == 0) {
        double* vir = R.q->vir;
        vir[0] += w * dx * dx;
        vir[1] += w * dy * dy;
        vir[2] += w * dx * dy;
        vir[3] += w * dy * dx;
        EdmdState* st = A.st;
        auto q = A.p + i;
        q->x = xi; q->y = yi; q->vx = vxi; q->vy = vyi; q->tl = t; q->coll = colli + 1;
        q = A.p + j;
        q->x = xj; q->y = yj; q->vx = vxj; q->vy = vyj; q->tl = t; q->coll = collj + 1;
        if (C.tape_cap > 0) {
            const int64_t k = st->ntape;
            if (k < C.tape_cap) {
                EdmdTapeRec rec;
                rec.t = t; rec.ax = dx; rec.ay = dy; rec.cx = dvx; rec.cy = dvy; rec.ff = ff;
                rec.i = i; rec.j = j; rec.g = 0;
                A.tape[k] = rec;
            }
            st->ntape = k + 1;
            st->wsum += w * (dx * dx + dy * dy);
            st->tlast = t;
        }
    }
    WAVE_SYNC();
    const Owner oi{i, xi, yi, vxi, vyi, ri, cxi, cyi};
    const Owner oj{j, xj, yj, vxj, vyj, rj, cxj, cyj};
    bool ov = false;
    double dti, dtj;
    int pi_, pj_;
    uint32_t cpi, cpj;
    predict_owners<false, W, (ML > 2 && !W)>(C, A, lane, t, 2, oi, oj, dti, pi_, cpi, dtj, pj_, cpj,
                                             ov, R.q->cand);
    flag_overlap(R, ov, i);
    double tci2, tcj2;
    int di, dj;
    cross_time<W>(C, t, xi, yi, vxi, vyi, cxi, cyi, tci2, di);
    cross_time<W>(C, t, xj, yj, vxj, vyj, cxj, cyj, tcj2, dj);
    const double tki = t + dti, tkj = t + dtj;
    /* insertion order, EDMD.c:3869-3879: crossings of i and j, then the
     * collisions of i and j */
    const int64_t rxi = take_rank(C, R, tci2);
    const int64_t rxj = take_rank(C, R, tcj2);
    const int64_t rki = take_rank(C, R, tki);
    const int64_t rkj = take_rank(C, R, tkj);
    if (lane == 0) {
        EdmdEv e;
        e.tcoll = tki; e.tcross = tci2; e.partner = pi_; e.cact = cpi; e.dir = di; e.pad = 0;
        A.e[i] = e;
        e.tcoll = tkj; e.tcross = tcj2; e.partner = pj_; e.cact = cpj; e.dir = dj;
        A.e[j] = e;
        A.erank[2 * i] = rki;
        A.erank[2 * i + 1] = rxi;
        A.erank[2 * j] = rkj;
        A.erank[2 * j + 1] = rxj;
    }
    path_update<ML>(C, A, lane, P, i, make_leaf(tki, rki, tci2, rxi, pi_, di), j,
                    make_leaf(tkj, rkj, tcj2, rxj, pj_, dj), R.q->top, R.t);
}

template <int ML, class AR>
__device__ __forceinline__ void ev_collision_grow(const EdmdConst& C, const AR& A, int lane, LoopRegs& R,
                                  int i, int j) {
    /* doTheCollisionGrow, EDMD.c:3465-3540 (2D): both disks fly with their
     * radii growing; the unit contact normal and the summed growth speed
     * enter the impulse; res and delta are the compile-time 1 and 0 of
     * EDMD.c:3467-3468; no virial. */
    const double delta = 0.1 * 0;
    const double res = 0.75 * 0 + 1;
    const EdmdEv ei = A.e[i];
    const int64_t rxi_old = A.erank[2 * i + 1]; /* crossing slot kept by a stale pop */
    const EdmdPart pi = A.p[i];
    const EdmdPart pj = A.p[j];
    const double vri = uni(A.vr[i]), vrj = uni(A.vr[j]);
    PathCache<ML> P;
    path_prefetch<ML>(C, A, lane, i, j, P);
    const double t = R.t;
    double xi = uni(pi.x), yi = uni(pi.y), vxi = uni(pi.vx), vyi = uni(pi.vy), tli = uni(pi.tl);
    double ri = uni(pi.rad);
    const double mi = uni(pi.m);
    const int cxi = uni((int)pi.cx), cyi = uni((int)pi.cy);
    const uint32_t colli = (uint32_t)uni((int)pi.coll);
    const uint32_t collj = (uint32_t)uni((int)pj.coll);
    const uint32_t ca = (uint32_t)uni((int)ei.cact);

    fly_grow(C, t, xi, yi, vxi, vyi, tli, ri, vri);
    xi = uni(xi);
    yi = uni(yi);
    ri = uni(ri);
    const bool valid = (ca == collj);
    trace_push(C, A, lane, t, EDMD_EV_COLLISION, i, j, valid ? 1 : 0);
    if (!valid) {
        if (lane == 0) {
            A.p[i].x = xi;
            A.p[i].y = yi;
            A.p[i].tl = t;
            A.p[i].rad = ri;
        }
        WAVE_SYNC();
        const Owner oi{i, xi, yi, vxi, vyi, ri, cxi, cyi, vri};
        bool ov = false;
        double dt, dtb;
        int pa, pb;
        uint32_t cpa, cpb;
        predict_owners<true>(C, A, lane, t, 1, oi, oi, dt, pa, cpa, dtb, pb, cpb, ov, R.q->cand);
        flag_overlap(R, ov, i);
        const double tk = t + dt;
        const double tci = uni(ei.tcross);
        const int64_t rci = uni64(rxi_old);
        const int diri = uni(ei.dir);
        const int64_t rk = take_rank(C, R, tk);
        if (lane == 0) {
            A.e[i].tcoll = tk;
            A.e[i].partner = pa;
            A.e[i].cact = cpa;
            A.erank[2 * i] = rk;
        }
        path_update<ML>(C, A, lane, P, i, make_leaf(tk, rk, tci, rci, pa, diri), -1, Leaf{}, R.q->top, R.t);
        return;
    }
    R.ncol++;
    double xj = uni(pj.x), yj = uni(pj.y), vxj = uni(pj.vx), vyj = uni(pj.vy), tlj = uni(pj.tl);
    double rj = uni(pj.rad);
    const double mj = uni(pj.m);
    const int cxj = uni((int)pj.cx), cyj = uni((int)pj.cy);
    fly_grow(C, t, xj, yj, vxj, vyj, tlj, rj, vrj);
    double dx = xj - xi;
    double dy = yj - yi;
    double dvx = vxj - vxi;
    double dvy = vyj - vyi;
    double dvr = vri + vrj;
    min_image(C, dx, dy);
    double dist = sqrt(dx * dx + dy * dy);
    double dxr = dx / dist;
    double dyr = dy / dist;
    double inv_mass = 1 / (mi + mj);
    double kernel = inv_mass * (1 + res) * (dxr * dvx + dyr * dvy - dvr);
    vxi = uni(vxi + (kernel * mj * dxr - 2 * mj * inv_mass * delta * dxr));
    vyi = uni(vyi + (kernel * mj * dyr - 2 * mj * inv_mass * delta * dyr));
    vxj = uni(vxj - (kernel * mi * dxr - 2 * mi * inv_mass * delta * dxr));
    vyj = uni(vyj - (kernel * mi * dyr - 2 * mi * inv_mass * delta * dyr));
    xj = uni(xj);
    yj = uni(yj);
    rj = uni(rj);
    if (lane == 0) {
        auto q = A.p + i;
        q->x = xi; q->y = yi; q->vx = vxi; q->vy = vyi; q->tl = t; q->rad = ri; q->coll = colli + 1;
        q = A.p + j;
        q->x = xj; q->y = yj; q->vx = vxj; q->vy = vyj; q->tl = t; q->rad = rj; q->coll = collj + 1;
    }
    WAVE_SYNC();
    const Owner oi{i, xi, yi, vxi, vyi, ri, cxi, cyi, vri};
    const Owner oj{j, xj, yj, vxj, vyj, rj, cxj, cyj, vrj};
    bool ov = false;
    double dti, dtj;
    int pi_, pj_;
    uint32_t cpi, cpj;
    predict_owners<true>(C, A, lane, t, 2, oi, oj, dti, pi_, cpi, dtj, pj_, cpj, ov, R.q->cand);
    flag_overlap(R, ov, i);
    double tci2, tcj2;
    int di, dj;
    cross_time<false>(C, t, xi, yi, vxi, vyi, cxi, cyi, tci2, di);
    cross_time<false>(C, t, xj, yj, vxj, vyj, cxj, cyj, tcj2, dj);
    const double tki = t + dti, tkj = t + dtj;
    /* insertion order, EDMD.c:3869-3879: crossings of i and j, then the
     * collisions of i and j */
    const int64_t rxi = take_rank(C, R, tci2);
    const int64_t rxj = take_rank(C, R, tcj2);
    const int64_t rki = take_rank(C, R, tki);
    const int64_t rkj = take_rank(C, R, tkj);
    if (lane == 0) {
        EdmdEv e;
        e.tcoll = tki; e.tcross = tci2; e.partner = pi_; e.cact = cpi; e.dir = di; e.pad = 0;
        A.e[i] = e;
        e.tcoll = tkj; e.tcross = tcj2; e.partner = pj_; e.cact = cpj; e.dir = dj;
        A.e[j] = e;
        A.erank[2 * i] = rki;
        A.erank[2 * i + 1] = rxi;
        A.erank[2 * j] = rkj;
        A.erank[2 * j + 1] = rxj;
    }
    path_update<ML>(C, A, lane, P, i, make_leaf(tki, rki, tci2, rxi, pi_, di), j,
                    make_leaf(tkj, rkj, tcj2, rxj, pj_, dj), R.q->top, R.t);
}

/* stopGrow, EDMD.c:4740-4785 (2D, no wells): final flight with growth, all
 * counters and image counters reset, normalizePhysicalQ (EDMD.c:5723-5764:
 * remove the mean momentum, scale to E/N = Einit), then the Normal
 * prediction of every disk with stopGrow's partner counters, and a new
 * calendar.  The caller continues in the Normal loop. */
template <bool W, class AR>
__device__ __forceinline__ bool ev_stop_grow(const EdmdConst& C, const AR& A, int lane,
                                             LoopRegs& R) {
    const double t = R.t;
    for (int q = lane; q < C.n; q += 64) {
        EdmdPart r = A.p[q];
        fly_grow(C, t, r.x, r.y, r.vx, r.vy, r.tl, r.rad, A.vr[q]);
        r.coll = 0;
        A.p[q] = r;
        A.img[2 * q] = 0;
        A.img[2 * q + 1] = 0;
    }
    WAVE_SYNC();
    const auto P = A.p;
    const int n = C.n;
    if (!(W && (C.walls & 4))) {
        const double px = ordered_sum(n, lane, [&](int q) { return P[q].vx * P[q].m; });
        const double py = ordered_sum(n, lane, [&](int q) { return P[q].vy * P[q].m; });
        for (int q = lane; q < n; q += 64) {
            const double m = P[q].m;
            P[q].vx -= px / (n * m);
            P[q].vy -= py / (n * m);
        }
    } else {
        /* in a circle, the angular momentum about the centre
         * (EDMD.c:5730-5749): dvT accumulates -m (x0 vy - y0 vx), dvM m r */
        const double h = C.halfLx;
        const double dvT = -ordered_sum(n, lane, [&](int q) {
            return P[q].m * (-P[q].vx * (P[q].y - h) + P[q].vy * (P[q].x - h));
        });
        const double dvM = ordered_sum(n, lane, [&](int q) {
            return P[q].m * sqrt((P[q].x - h) * (P[q].x - h) + (P[q].y - h) * (P[q].y - h));
        });
        const double dv = dvT / dvM;
        for (int q = lane; q < n; q += 64) {
            const double x0 = P[q].x - h, y0 = P[q].y - h;
            const double r = sqrt(x0 * x0 + y0 * y0);
            P[q].vx += -dv * y0 / r;
            P[q].vy += dv * x0 / r;
        }
    }
    WAVE_SYNC();
    const double E = ordered_sum(n, lane, [&](int q) {
        double a = P[q].vx;
        return 0.5 * P[q].m * (a * a + P[q].vy * P[q].vy);
    });
    for (int q = lane; q < n; q += 64) {
        P[q].vx /= sqrt(E / n / C.einit);
        P[q].vy /= sqrt(E / n / C.einit);
        P[q].coll = 1;
    }
    WAVE_SYNC();
    bool ov = false;
    /* per particle: collision, then crossing (EDMD.c:4770-4776) */
    for (int q = lane; q < n; q += 64)
        ov |= sweep_one<false, W>(C, A, t, q, R.paul, R.ctr + 2 * (int64_t)q + 1,
                               R.ctr + 2 * (int64_t)q, true);
    R.ctr += 2 * (int64_t)n;
    WAVE_SYNC();
    const bool any_ov = __ballot(ov) != 0ull;
    rebuild_tree(C, A, lane);
    top_load(C, A, lane, R.q->top);
    if (lane == 0) {
        A.st->growing = 0;
        A.st->next_grow = INF_D;
    }
    WAVE_SYNC();
    return any_ov;
}

template <int ML, bool G, bool W, class AR>
__device__ __forceinline__ void ev_single(const EdmdConst& C, const AR& A, int lane, LoopRegs& R, int p,
                          int d) {
    /* The events that change one disk.  d = 1-4: a cell crossing in that
     * direction (doTheCrossing, EDMD.c:2501-2590; its freeFly is the
     * dispatch pointer, freeFlyGrow while growing).  d = 5 + xy: a wall hit
     * (doTheWallNormal, EDMD.c:3384-3460, without thermal or shear walls;
     * doTheWallGrow while growing): counted as a collision, the momentum
     * given to the wall accumulated for the thermo row, the normal velocity
     * reversed times resW and the tangential one scaled by resT, a flat
     * wall's hit written to the tape when taping.  Both then predict the
     * crossing slot and the collision slot again, in that order. */
    const bool wall = W && d >= 5;
    const EdmdPart pp = A.p[p];
    const double gvr = G ? uni(A.vr[p]) : 0.0;
    PathCache<ML> P;
    path_prefetch<ML>(C, A, lane, p, -1, P);
    const double t = R.t;
    double x = uni(pp.x), y = uni(pp.y), tl = uni(pp.tl);
    double vx = uni(pp.vx), vy = uni(pp.vy);
    double r = uni(pp.rad);
    int cx = uni((int)pp.cx), cy = uni((int)pp.cy);
    trace_push(C, A, lane, t, wall ? EDMD_EV_WALL : EDMD_EV_CELLCROSS, p, wall ? d - 5 : d, 1);
    if (G) {
        fly_grow(C, t, x, y, vx, vy, tl, r, gvr);
        r = uni(r);
    } else {
        fly_v<W>(C, t, x, y, vx, vy, tl);
    }
    x = uni(x);
    y = uni(y);
    vx = uni(vx);
    vy = uni(vy);

    if (wall && G) {
        /* doTheWallGrow, EDMD.c:3333-3382: a collision, no momentum to the
         * wall; the normal velocity turned away with 2 vr added (for y,
         * which way by the disk's height) */
        R.ncol++;
        if (d == 5) {
            const double sg = vx < 0 ? -1.0 : (vx > 0 ? 1.0 : 0.0);
            vx = -sg * (fabs(vx) + 2 * gvr);
        } else if (d == 6) {
            if (y > C.Ly - 3) vy = -vy - 2 * gvr;
            else vy = -vy + 2 * gvr;
        } else {
            /* the circle: reflected about the normal, 2 vr added along it */
            double nx, ny;
            edmd_sincos(edmd_atan2(y - C.halfLx, x - C.halfLx), ny, nx);
            const double mix = -(1 + C.res_wall) * (vx * nx + vy * ny);
            vx += (mix - 2 * gvr) * nx;
            vy += (mix - 2 * gvr) * ny;
        }
        vx = uni(vx);
        vy = uni(vy);
        if (lane == 0) {
            const auto q = A.p + p;
            q->x = x;
            q->y = y;
            q->tl = tl;
            q->vx = vx;
            q->vy = vy;
            q->rad = r;
            q->coll = pp.coll + 1;
        }
        WAVE_SYNC();
    } else if (wall) {
        R.ncol++;
        const double m = uni(pp.m);
        double dp;
        /* the tangential product is made +0.0 where it is -0.0 (resT = 0
         * times a negative velocity): the reference's crossing prediction
         * divides by a -0.0 velocity and flies the disk to t = -inf */
        double dpl = 0, dpm = 0, dpr = 0;
        const double vx0 = vx, vy0 = vy; /* before the hit, for the tape */
        if (d == 5) {
            dp = fabs((C.res_wall + 1) * m * vx);
            if (C.walls & 8) {
                /* EDMD.c:3393-3409: the side walls within 3 of the box's edges */
                if (vx < 0) {
                    if (x - 3 < 0) dpl = dp;
                    else dpm = dp;
                } else {
                    if (x + 3 > C.Lx) dpr = dp;
                    else dpm = dp;
                }
            }
            if (C.thermal_wall) {
                /* thermoWall (EDMD.c:3411-3413): the normal speed drawn */
                vx = -ref_sign(vx) * mt_drand0(A, lane, C.temperature / m);
            } else {
                vx = -C.res_wall * vx;
                vy = C.res_tan * vy + 0.0;
            }
        } else if (d == 6) {
            dp = fabs((C.res_wall + 1) * m * vy);
            if (C.thermal_wall) {
                vy = -ref_sign(vy) * mt_drand0(A, lane, C.temperature / m);
            } else {
                vy = -C.res_wall * vy;
                vx = C.res_tan * vx + 0.0;
            }
            /* addShearWall (EDMD.c:3429-3439, without the delta model's
             * kick): the top wall drives +0.1 along x, the bottom -0.1 */
            if (C.shear_wall) vx = (y + 2 * r > C.Ly) ? 0.1 : -0.1;
        } else {
            /* the circle (EDMD.c:3441-3454): the normal velocity reversed
             * times resW (thermal: both components drawn), |m mix| to the
             * wall */
            double nx, ny;
            edmd_sincos(edmd_atan2(y - C.halfLx, x - C.halfLx), ny, nx);
            const double mix = -(1 + C.res_wall) * (vx * nx + vy * ny);
            if (C.thermal_wall) {
                vx = -nx * mt_drand0(A, lane, C.temperature);
                vy = -ny * mt_drand0(A, lane, C.temperature);
            } else {
                vx += mix * nx;
                vy += mix * ny;
            }
            dp = fabs(m * mix);
        }
        vx = uni(vx);
        vy = uni(vy);
        if (lane == 0) {
            A.st->dpw += dp;
            if (C.walls & 8) {
                A.st->dpl += dpl;
                A.st->dpm += dpm;
                A.st->dpr += dpr;
            }
            if (C.tape_cap > 0 && d != 7) {
                /* a flat wall's record: j = -1 - xy, the normal and
                 * tangential velocities before the hit, resW, resT and the
                 * contact coordinate */
                EdmdState* st = A.st;
                const int64_t k = st->ntape;
                if (k < C.tape_cap) {
                    EdmdTapeRec rec;
                    rec.t = t;
                    rec.ax = d == 5 ? vx0 : vy0;
                    rec.ay = d == 5 ? vy0 : vx0;
                    rec.cx = C.res_wall;
                    rec.cy = C.res_tan;
                    rec.ff = d == 5 ? x : y;
                    rec.i = p;
                    rec.j = d == 5 ? -1 : -2;
                    rec.g = C.field_on ? C.field : 0.0;
                    A.tape[k] = rec;
                }
                st->ntape = k + 1;
            }
            const auto q = A.p + p;
            q->x = x;
            q->y = y;
            q->tl = tl;
            q->vx = vx;
            q->vy = vy;
            q->coll = pp.coll + 1;
        }
        WAVE_SYNC();
    } else {
        /* removeFromCell: drop p, keeping the order of the others */
        const int c0 = cy * C.ncx + cx;
        const int n0 = A.ccnt[c0];
        int v = (lane < n0) ? A.cslot[(size_t)c0 * C.cap + lane] : -1;
        uint64_t hit = __ballot(v == p);
        int pos = hit ? (int)__builtin_ctzll(hit) : n0;
        if (lane > pos && lane < n0) A.cslot[(size_t)c0 * C.cap + lane - 1] = v;
        if (lane == 0) A.ccnt[c0] = n0 - 1;

        int wx = 0, wy = 0; /* periodic image change */
        switch (d) {
            case 1:
                if (cx - 1 == -1) { cx = C.ncx - 1; wx = -1; } else cx -= 1;
                break;
            case 2:
                if (cx + 1 == C.ncx) { cx = 0; wx = 1; } else cx += 1;
                break;
            case 3:
                if (cy - 1 == -1) { cy = C.ncy - 1; wy = -1; } else cy -= 1;
                break;
            default:
                if (cy + 1 == C.ncy) { cy = 0; wy = 1; } else cy += 1;
                break;
        }
        WAVE_SYNC();
        const int c1 = cy * C.ncx + cx;
        const int n1 = A.ccnt[c1];
        if (n1 >= C.cap) {
            if (R.status == EDMD_DEV_OK) {
                R.status = EDMD_DEV_CELL_OVERFLOW;
                R.err_i = p;
                R.err_j = c1;
            }
            return;
        }
        if (lane == 0) {
            A.cslot[(size_t)c1 * C.cap + n1] = p; /* newest entry: visited first */
            A.ccnt[c1] = n1 + 1;
            const auto q = A.p + p;
            q->x = x;
            q->y = y;
            q->tl = tl;
            if (W) { /* changed by the flight under the field or damping */
                q->vx = vx;
                q->vy = vy;
            }
            if (G) q->rad = r;
            q->cx = (int16_t)cx;
            q->cy = (int16_t)cy;
            if (wx) A.img[2 * p] += wx;
            if (wy) A.img[2 * p + 1] += wy;
        }
        WAVE_SYNC();
    }
    const Owner o{p, x, y, vx, vy, r, cx, cy, gvr};
    bool ov = false;
    double dt, dtb;
    int pa, pb;
    uint32_t cpa, cpb;
    predict_owners<G, W, (ML > 2 && !W)>(C, A, lane, t, 1, o, o, dt, pa, cpa, dtb, pb, cpb, ov,
                                         R.q->cand);
    flag_overlap(R, ov, p);
    double tc;
    int dir;
    cross_time<W && !G>(C, t, x, y, vx, vy, cx, cy, tc, dir);
    const double tk = t + dt;
    /* crossingEvent(i), then collisionEvent(i), EDMD.c:2587-2589, 3458-3459 */
    const int64_t rx = take_rank(C, R, tc);
    const int64_t rk = take_rank(C, R, tk);
    if (lane == 0) {
        EdmdEv e;
        e.tcoll = tk; e.tcross = tc; e.partner = pa; e.cact = cpa; e.dir = dir; e.pad = 0;
        A.e[p] = e;
        A.erank[2 * p] = rk;
        A.erank[2 * p + 1] = rx;
    }
    path_update<ML>(C, A, lane, P, p, make_leaf(tk, rk, tc, rx, pa, dir), -1, Leaf{}, R.q->top, R.t);
}

/* Persistent event loop of one system on one wavefront; ML bounds the
 * calendar depth of every system in the launch.  A holds the system's arrays
 * in HBM (EdmdArrays) or in LDS (EdmdArraysL); the caller has checked that
 * the system's growth phase matches G. */
template <int ML, bool G, bool W, int WPB = 1, class AR>
__device__ __forceinline__ void run_loop(const EdmdConst& C, const AR& A, EdmdRunArgs ra) {
    /* WPB wavefronts per workgroup, each looping over its own system with
     * its own LDS queue state */
    const int lane = threadIdx.x & 63;
    EdmdState* st = A.st;
    __shared__ QueueState Qs[WPB];
    LoopRegs R;
    R.q = &Qs[WPB > 1 ? wave_in_group() : 0];
    R.t = uni(st->t);
    R.ncol = st->ncol;
    R.nevents = st->nevents;
    R.status = st->status;
    R.err_i = st->err_i;
    R.err_j = st->err_j;
    R.paul = uni(st->paul);
    R.ctr = uni64(st->ctr);
    R.win = uni64(st->win);
    R.cur = uni((int)(R.win % C.nlists));
    if (lane == 0)
        for (int k = 0; k < 4; ++k) R.q->vir[k] = st->vir[k];
    next_special(st, R);
    top_load(C, A, lane, R.q->top);
    uint64_t ncross = st->ncross;
    int reason = EDMD_STOP_NONE;
    int last_type = st->last_type;

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
            const int sp = R.special;
            R.t = R.next_special;
            trace_push(C, A, lane, R.t, sp, 0, 0, 1);
            if (sp == EDMD_EV_SCREENSHOT) {
                ev_screenshot<G, W>(C, A, lane, R);
            } else if (sp == EDMD_EV_THERMO) {
                ev_thermo(C, A, lane, R);
            } else if (sp == EDMD_EV_GROWSTOP) {
                if (G) {
                    flag_overlap(R, ev_stop_grow<W>(C, A, lane, R), 0);
                    R.ncol = 0; /* stopGrow resets ncol and ncross, EDMD.c:4745-4746 */
                    ncross = 0;
                }
            } else {
                if (ev_rescale<G, W>(C, A, lane, R) && R.status == EDMD_DEV_OK)
                    R.status = EDMD_DEV_OVERLAP;
            }
            next_special(st, R);
            R.nevents++;
            last_type = sp;
            if (G && sp == EDMD_EV_GROWSTOP) { reason = EDMD_STOP_GROWN; break; }
            if (ra.stop_mask & (1 << sp)) { reason = EDMD_STOP_SPECIAL; break; }
            continue;
        }
        R.t = key;
        if (aux >= 0) {
            if (G) ev_collision_grow<ML>(C, A, lane, R, p, aux);
            else ev_collision<ML, W>(C, A, lane, R, p, aux);
            last_type = EDMD_EV_COLLISION;
        } else {
            /* a crossing (code -1..-4) or a wall hit (-5 - xy) */
            const bool wall = W && aux <= EDMD_WALL_CODE(0);
            ev_single<ML, G, W>(C, A, lane, R, p, wall ? 5 + EDMD_WALL_CODE(0) - aux : -aux);
            if (wall) {
                last_type = EDMD_EV_WALL;
            } else {
                ncross++;
                last_type = EDMD_EV_CELLCROSS;
            }
        }
        R.nevents++;
        if (ra.stop_mask & (1 << last_type)) { reason = EDMD_STOP_SPECIAL; break; }
    }

    if (lane == 0) {
        st->t = R.t;
        st->ncol = R.ncol;
        st->ncross = ncross;
        st->nevents = R.nevents;
        st->status = R.status;
        st->err_i = R.err_i;
        st->err_j = R.err_j;
        st->stop_reason = reason;
        st->last_type = last_type;
        st->paul = R.paul;
        st->ctr = R.ctr;
        st->win = R.win;
        for (int k = 0; k < 4; ++k) st->vir[k] = R.q->vir[k];
    }
    top_store(C, A, lane, R.q->top);
}

#endif
