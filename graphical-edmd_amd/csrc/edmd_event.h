/*
 * One particle event in steps, shared by the event loops: event_open (records
 * read, free flight, collision rule, cell or wall change) and event_predict
 * (new collision and crossing times), which write nothing to the system
 * (event_predict only where SPEC is false, the neighbours' flights under the
 * field or damping), then event_cells, event_store, event_enter, event_sums and
 * event_slots, which do.
 *
 * Half-wave layout: lanes 0-31 hold the event's first disk, lanes 32-63 its
 * second one (a valid collision's partner; else the first disk again), so
 * flights, crossing times, ranks, leaves and record writes of both disks
 * are one instruction stream, and each half scans its own disk's
 * neighbours.  Values of the other half come by v_permlane32_swap.  Before,
 * every lane computed both disks' values one after the other: 594 vector and
 * 407 scalar instructions per event of the 4096-replica batch and 15.6 vector
 * writes, 120.1 ms a launch; now 632, 331 and 9.4, 106.5 ms.
 *
 * Reference line numbers are those of src/EDMD.c.
 */
#ifndef EDMD_EVENT_H
#define EDMD_EVENT_H

#include "edmd_device.h"

/* v of lanes 0-31 (a) and of lanes 32-63 (b), on every lane's counterpart in
 * the other half too: lane l gets v of lanes l & 31 and 32 + (l & 31). */
__device__ __forceinline__ void halves(int v, int& a, int& b) {
    const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    a = (int)r[0];
    b = (int)r[1];
}

__device__ __forceinline__ void halves(double v, double& a, double& b) {
    const long long q = __double_as_longlong(v);
    int al, bl, ah, bh;
    halves((int)q, al, bl);
    halves((int)(q >> 32), ah, bh);
    a = __longlong_as_double(((long long)ah << 32) | (unsigned int)al);
    b = __longlong_as_double(((long long)bh << 32) | (unsigned int)bl);
}

/* v of the other half's counterpart lane, through the LDS crossbar: one
 * instruction a word and none of the vector unit's, whose issue bounds the
 * batched loop (a swap takes two moves and the swap). */
__device__ __forceinline__ int other_half(int v, int lane) {
    return __builtin_amdgcn_ds_bpermute(4 * (lane ^ 32), v);
}

__device__ __forceinline__ double other_half(double v, int lane) {
    const long long q = __double_as_longlong(v);
    const int lo = other_half((int)q, lane), hi = other_half((int)(q >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

/* v of the two rows of 16 lanes of each half, on both: a from the even row,
 * b from the odd one. */
__device__ __forceinline__ void rows(double v, double& a, double& b) {
    const long long q = __double_as_longlong(v);
    const auto l = __builtin_amdgcn_permlane16_swap((unsigned)q, (unsigned)q, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap((unsigned)(q >> 32), (unsigned)(q >> 32), false, false);
    a = __longlong_as_double(((long long)h[0] << 32) | l[0]);
    b = __longlong_as_double(((long long)h[1] << 32) | l[1]);
}

/* The smaller of two numbers, neither NaN, in one instruction (a select
 * takes a comparison and two moves). */
__device__ __forceinline__ double min_f64(double a, double b) {
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

/* Minimum over each half (32 lanes), on all its lanes. */
__device__ __forceinline__ double half_min(double v) {
    v = min_f64(v, dpp_f64<0xb1>(v));
    v = min_f64(v, dpp_f64<0x4e>(v));
    v = min_f64(v, dpp_f64<0x141>(v));
    v = min_f64(v, dpp_f64<0x140>(v));
    double a, b;
    rows(v, a, b);
    return min_f64(a, b);
}

__device__ __forceinline__ double flip_if(double v, bool neg) {
    return __longlong_as_double(__double_as_longlong(v) ^ ((long long)neg << 63));
}

enum { EVK_STALE, EVK_COLLISION, EVK_CROSSING, EVK_WALL };

/* An event being handled.  Fields marked (h) differ between the halves. */
struct EvState {
    int own;               /* (h) disk */
    double x, y, vx, vy;   /* (h) its state at t, after the event */
    double r, m, vr;       /* (h) radius, mass, growth rate */
    uint32_t coll;         /* (h) its collision counter after the event */
    int cx, cy;            /* (h) its cell after the event */
    double tk, tc;         /* (h) absolute times of the next collision and crossing */
    int partner, dir;      /* (h) */
    uint32_t cact;         /* (h) partner's counter */
    int kind, nown;        /* EVK_*, disks that change: 1 or 2 */
    int totA, totB;        /* candidates staged for each disk */
    bool ov;               /* an overlap was seen (per lane) */
    bool none0;            /* a disk without a candidate: partner 0's counter was read */
    int64_t rx_old;        /* rank of the crossing slot a stale event keeps */
    /* collision: contact vector, relative velocity before, impulse, virial weight */
    double dx, dy, dvx, dvy, ff, w;
    /* crossing: direction, the cell left, its count and (by lane) its slots */
    int d, c0, n0, slot, n1;
    /* wall: momentum to the wall (total, left, mid, right), velocity before */
    double dp, dpl, dpm, dpr, vx0, vy0;
};

/* Reads the event's records and applies its rule in registers: p's leaf
 * holds key t and event code aux (the partner, or minus a direction, or a
 * wall code). */
template <bool G, bool W, class AR>
__device__ __forceinline__ void event_open(const EdmdConst& C, const AR& A, int lane, double t,
                                           int p, int aux, EvState& S) {
    const bool hi = lane >= 32;
    const bool pair = aux >= 0;
    S.own = (pair && hi) ? aux : p;
    const EdmdPart rec = A.p[S.own];
    S.vr = G ? A.vr[S.own] : 0.0;
    EdmdEv ei;
    S.rx_old = 0;
    if (pair) {
        ei = A.e[p];
        S.rx_old = A.erank[2 * p + 1]; /* crossing slot kept by a stale pop */
    }
    S.x = rec.x;
    S.y = rec.y;
    S.vx = rec.vx;
    S.vy = rec.vy;
    S.r = rec.rad;
    S.m = rec.m;
    S.coll = rec.coll;
    S.cx = rec.cx;
    S.cy = rec.cy;
    S.ov = false;
    S.nown = 1;
    double tl = rec.tl;
    if (G) fly_grow(C, t, S.x, S.y, S.vx, S.vy, tl, S.r, S.vr);
    else fly_v<W>(C, t, S.x, S.y, S.vx, S.vy, tl);

    if (pair) {
        const uint32_t collj = (uint32_t)__builtin_amdgcn_readlane((int)S.coll, 32);
        const bool valid = __builtin_amdgcn_readfirstlane((int)ei.cact) == (int)collj;
        S.tc = ei.tcross;
        S.dir = ei.dir;
        if (!valid) {
            /* stale prediction: free flight of i and a new collision slot;
             * the upper half takes i's values */
            S.kind = EVK_STALE;
            S.own = p;
            int u;
            double g;
            halves(S.x, S.x, g);
            halves(S.y, S.y, g);
            halves(S.vx, S.vx, g);
            halves(S.vy, S.vy, g);
            halves(S.r, S.r, g);
            halves(S.m, S.m, g);
            halves(S.cx, S.cx, u);
            halves(S.cy, S.cy, u);
            int c;
            halves((int)S.coll, c, u);
            S.coll = (uint32_t)c;
            if (G) halves(S.vr, S.vr, g);
            return;
        }
        S.kind = EVK_COLLISION;
        S.nown = 2;
        S.coll = S.coll + 1;
        /* differences in the order j - i on both halves */
        S.dx = flip_if(other_half(S.x, lane) - S.x, hi);
        S.dy = flip_if(other_half(S.y, lane) - S.y, hi);
        S.dvx = flip_if(other_half(S.vx, lane) - S.vx, hi);
        S.dvy = flip_if(other_half(S.vy, lane) - S.vy, hi);
        const double mo = other_half(S.m, lane); /* the other disk's mass */
        const double inv_mass = 1 / (S.m + mo);
        min_image(C, S.dx, S.dy);
        if (!G) {
            /* doTheCollisionNormal, EDMD.c:3583-3606, 3802-3827 */
            const double kernel = inv_mass * (1 + C.res) * (S.dx * S.dvx + S.dy * S.dvy);
            const double ro = other_half(S.r, lane);
            S.ff = kernel / (4 * (hi ? ro : S.r) * (hi ? S.r : ro));
            S.w = S.m * mo * S.ff;
            S.vx = S.vx + flip_if(S.ff * mo * S.dx, hi);
            S.vy = S.vy + flip_if(S.ff * mo * S.dy, hi);
        } else {
            /* doTheCollisionGrow, EDMD.c:3465-3540 (2D): the unit contact
             * normal and the summed growth speed enter the impulse; res and
             * delta are the compile-time 1 and 0 of EDMD.c:3467-3468; no
             * virial */
            const double delta = 0.1 * 0;
            const double res = 0.75 * 0 + 1;
            const double dvr = S.vr + other_half(S.vr, lane);
            const double dist = sqrt(S.dx * S.dx + S.dy * S.dy);
            const double dxr = S.dx / dist;
            const double dyr = S.dy / dist;
            const double kernel = inv_mass * (1 + res) * (dxr * S.dvx + dyr * S.dvy - dvr);
            S.vx = S.vx + flip_if(kernel * mo * dxr - 2 * mo * inv_mass * delta * dxr, hi);
            S.vy = S.vy + flip_if(kernel * mo * dyr - 2 * mo * inv_mass * delta * dyr, hi);
        }
        return;
    }
    if (W && aux <= EDMD_WALL_CODE(0)) {
        /* doTheWallNormal (EDMD.c:3384-3460; counted as a collision, the
         * momentum given to the wall accumulated for the thermo row, the
         * normal velocity reversed times resW and the tangential one scaled
         * by resT) or doTheWallGrow while growing (EDMD.c:3333-3382: no
         * momentum to the wall; the normal velocity turned away with 2 vr
         * added, for y which way by the disk's height) */
        S.kind = EVK_WALL;
        S.d = EDMD_WALL_CODE(0) - aux; /* 0: normal to x, 1: normal to y, 2: the circle */
        S.coll = S.coll + 1;
        S.vx0 = S.vx;
        S.vy0 = S.vy;
        S.dp = S.dpl = S.dpm = S.dpr = 0;
        const double x = S.x, y = S.y;
        double vx = S.vx, vy = S.vy;
        if (G) {
            if (S.d == 0) {
                const double sg = vx < 0 ? -1.0 : (vx > 0 ? 1.0 : 0.0);
                vx = -sg * (fabs(vx) + 2 * S.vr);
            } else if (S.d == 1) {
                if (y > C.Ly - 3) vy = -vy - 2 * S.vr;
                else vy = -vy + 2 * S.vr;
            } else {
                /* the circle: reflected about the normal, 2 vr added along it */
                const double2 nrm = circle_normal(y - C.halfLx, x - C.halfLx);
                const double nx = nrm.x, ny = nrm.y;
                const double mix = -(1 + C.res_wall) * (vx * nx + vy * ny);
                vx += (mix - 2 * S.vr) * nx;
                vy += (mix - 2 * S.vr) * ny;
            }
        } else {
            const double m = S.m;
            /* the tangential product is made +0.0 where it is -0.0 (resT = 0
             * times a negative velocity): the reference's crossing
             * prediction divides by a -0.0 velocity and flies the disk to
             * t = -inf */
            if (S.d == 0) {
                S.dp = fabs((C.res_wall + 1) * m * vx);
                if (C.walls & 8) {
                    /* EDMD.c:3393-3409: the side walls within 3 of the box's edges */
                    if (vx < 0) {
                        if (x - 3 < 0) S.dpl = S.dp;
                        else S.dpm = S.dp;
                    } else {
                        if (x + 3 > C.Lx) S.dpr = S.dp;
                        else S.dpm = S.dp;
                    }
                }
                if (C.thermal_wall) {
                    /* thermoWall (EDMD.c:3411-3413): the normal speed drawn */
                    vx = -ref_sign(vx) * mt_drand0(A, lane, C.temperature / m);
                } else {
                    vx = -C.res_wall * vx;
                    vy = C.res_tan * vy + 0.0;
                }
            } else if (S.d == 1) {
                S.dp = fabs((C.res_wall + 1) * m * vy);
                if (C.thermal_wall) {
                    vy = -ref_sign(vy) * mt_drand0(A, lane, C.temperature / m);
                } else {
                    vy = -C.res_wall * vy;
                    vx = C.res_tan * vx + 0.0;
                }
                /* addShearWall (EDMD.c:3429-3439, without the delta model's
                 * kick): the top wall drives +0.1 along x, the bottom -0.1 */
                if (C.shear_wall) vx = (y + 2 * S.r > C.Ly) ? 0.1 : -0.1;
            } else {
                /* the circle (EDMD.c:3441-3454): the normal velocity reversed
                 * times resW (thermal: both components drawn), |m mix| to the
                 * wall */
                const double2 nrm = circle_normal(y - C.halfLx, x - C.halfLx);
                const double nx = nrm.x, ny = nrm.y;
                const double mix = -(1 + C.res_wall) * (vx * nx + vy * ny);
                if (C.thermal_wall) {
                    vx = -nx * mt_drand0(A, lane, C.temperature);
                    vy = -ny * mt_drand0(A, lane, C.temperature);
                } else {
                    vx += mix * nx;
                    vy += mix * ny;
                }
                S.dp = fabs(m * mix);
            }
        }
        S.vx = vx;
        S.vy = vy;
        return;
    }
    /* doTheCrossing, EDMD.c:2501-2590: the cell left (removeFromCell) is
     * read now and edited at the commit; the scan of the new neighbourhood
     * skips the disk itself, so both orders list the same candidates */
    S.kind = EVK_CROSSING;
    S.d = -aux;
    S.c0 = S.cy * C.ncx + S.cx;
    S.n0 = A.ccnt[S.c0];
    S.slot = lane < C.cap ? A.cslot[(size_t)S.c0 * C.cap + lane] : -1;
    switch (S.d) {
        case 1: S.cx = S.cx - 1 == -1 ? C.ncx - 1 : S.cx - 1; break;
        case 2: S.cx = S.cx + 1 == C.ncx ? 0 : S.cx + 1; break;
        case 3: S.cy = S.cy - 1 == -1 ? C.ncy - 1 : S.cy - 1; break;
        default: S.cy = S.cy + 1 == C.ncy ? 0 : S.cy + 1; break;
    }
}

/* Crossing time of each half's disk (crossingEventNormal, EDMD.c:2405-2482,
 * without field or damping): the even row of 16 lanes takes the x axis, the
 * odd one the y axis, so both edges' times of both disks are one division. */
__device__ __forceinline__ void cross_rows(const EdmdConst& C, int lane, double t,
                                           const EvState& S, double& tout, int& dir) {
    const bool ax = (lane & 16) != 0;
    const double v = ax ? S.vy : S.vx;
    const bool neg = v < 0;
    const int c = (ax ? S.cy : S.cx) + (neg ? 0 : 1);
    const double edge = wrap_inside(c * (ax ? C.csy : C.csx) - (ax ? S.y : S.x),
                                    ax ? C.halfLy : C.halfLx, ax ? C.Ly : C.Lx);
    double tx, ty;
    rows(edge / v, tx, ty);
    if (tx < ty) {
        tout = t + tx;
        dir = S.vx < 0 ? 1 : 2;
    } else {
        tout = t + ty;
        dir = S.vy < 0 ? 3 : 4;
    }
}

/* Whether the neighbour scan below stages this cell capacity in LDS. */
__device__ __forceinline__ bool staged_cap(const EdmdConst& C) {
    return C.cap <= EDMD_STAGE_CAP && (C.cap & 3) == 0;
}

/* Next collision of the disks of an event (collisionEventNormal / Grow,
 * EDMD.c:2829-3003, 3104-3230).
 *
 * Lane e < 9 of each half reads cell e of its disk's 3x3 block (y offset
 * outer, x offset inner): its count and its whole slot row in one round
 * trip.  A scan over the counts places every candidate at its traversal
 * position in the half's LDS stage, each cell's newest entry first
 * (EDMD.c:2959-3003).  Two disks: lane f of a half evaluates its disk's
 * candidates f, f + 32, ...; one disk: all 64 lanes its f, f + 64, ....
 * Each lane keeps its first strictly least time, and the least over the
 * half, the lowest position among equal times, is the reference's
 * strict-less first minimum.  Of cell capacities that the stage cannot take
 * (over EDMD_STAGE_CAP, or rows that are not whole 16-byte chunks) each lane
 * reads its candidate's slot from memory: one round trip more a pass.
 *
 * SPEC = false: the event's records are stored already (event_store), and
 * the field's or the damping's flights of the neighbours (EDMD.c:2664-2666)
 * are stored here.  SPEC = true: nothing is written; the other disk of a
 * collision appears among the candidates with its state before the event,
 * and its new one, in the other half's registers, takes its place. */
__device__ __forceinline__ int near_cell(const EdmdConst& C, int cx, int cy, int e) {
    const int ey = (e * 11) >> 5; /* e / 3 */
    return wrap_cell(cy + ey - 1, C.ncy) * C.ncx + wrap_cell(cx + (e - 3 * ey) - 1, C.ncx);
}

template <bool G, bool W, bool SPEC, class AR>
__device__ __forceinline__ void predict_halves(const EdmdConst& C, const AR& A, int lane, double t,
                                               EvState& S, double& dt, int32_t* stage) {
    const bool hi = lane >= 32;
    const int sub = lane & 31;
    const bool two = S.nown == 2;
    const bool staged = SPEC || staged_cap(C);
    const bool ent = sub < 9 && (two || !hi);
    int cnt = 0;
    int4 row[EDMD_STAGE_CAP / 4];
    if (ent) {
        const int cell = near_cell(C, S.cx, S.cy, sub);
        const int4* src = (const int4*)(A.cslot + (int64_t)cell * C.cap);
        cnt = A.ccnt[cell];
        if (staged) {
#pragma unroll
            for (int c = 0; c < EDMD_STAGE_CAP / 4; ++c)
                if (4 * c < C.cap) row[c] = src[c];
        }
    }
    /* the other disk's state, for its place among the candidates */
    int oth = -1;
    double xo = 0, yo = 0, vxo = 0, vyo = 0, ro = 0;
    uint32_t co = 0;
    if (SPEC && two) {
        oth = other_half(S.own, lane);
        co = (uint32_t)other_half((int)S.coll, lane);
        xo = other_half(S.x, lane);
        yo = other_half(S.y, lane);
        vxo = other_half(S.vx, lane);
        vyo = other_half(S.vy, lane);
        if (G) ro = other_half(S.r, lane);
    }
    int incl = cnt; /* inclusive scan within the row of 16 lanes */
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xf, 0xf, true);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xf, 0xf, true);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xf, 0xf, true);
    incl += __builtin_amdgcn_update_dpp(0, incl, 0x118, 0xf, 0xf, true);
    const int totA = __builtin_amdgcn_readlane(incl, 8);
    const int totB = two ? __builtin_amdgcn_readlane(incl, 40) : 0;
    S.totA = totA;
    S.totB = totB;
    S.n1 = __builtin_amdgcn_readlane(cnt, 4); /* the disk's own cell */
    int32_t* const half_stage =
        stage + ((two && hi) ? EDMD_STAGE_HALF : 0) + EDMD_STAGE_CAP;
    if (!staged) {
        if (ent) {
            /* what the fetch below needs of this cell: the candidates up to
             * its last, and the slot that candidate 0 would have */
            const int64_t at = (int64_t)near_cell(C, S.cx, S.cy, sub) * C.cap + incl - 1;
            half_stage[sub] = incl;
            half_stage[16 + 2 * sub] = (int)at;
            half_stage[17 + 2 * sub] = (int)(at >> 32);
        }
    } else if (ent && cnt > 0) {
        /* slot k (k-th oldest) goes to incl - 1 - k.  The row is written
         * whole, its last slot first: an unused slot (k >= cnt) falls on the
         * slot k - cnt, or a lower one, of a cell before, which is written
         * after it, or on the room before the stage; so no slot needs a test */
        int32_t* const at = half_stage + incl - EDMD_STAGE_CAP;
#pragma unroll
        for (int c = EDMD_STAGE_CAP / 4 - 1; c >= 0; --c) {
            if (4 * c >= C.cap) continue;
            const int v[4] = {row[c].x, row[c].y, row[c].z, row[c].w};
#pragma unroll
            for (int k = 3; k >= 0; --k) {
                at[EDMD_STAGE_CAP - 1 - 4 * c - k] = v[k];
                asm volatile("" ::: "memory"); /* one write each, in this order */
            }
        }
    }
    WAVE_SYNC();
    const double lim = G ? EDMD_GROW_NONE : EDMD_NEVER;
    const int most = totA > totB ? totA : totB;
    const int mine = (two && hi) ? totB : totA;
    const int li = two ? sub : lane, step = two ? 32 : 64;
    const int passes = (most + step - 1) / step;
    double bt = INF_D;
    int bq = 0, bf = 0;
    uint32_t bc = 0;
    for (int pass = 0; pass < passes; ++pass) {
        const int f = pass * step + li;
        int q = -1;
        if (f < mine) {
            if (staged) {
                q = half_stage[f];
            } else {
                int e = 0; /* the candidate's cell */
#pragma unroll
                for (int s = 0; s < 8; ++s) e += f >= half_stage[s] ? 1 : 0;
                const int64_t at = (int64_t)((uint64_t)(uint32_t)half_stage[17 + 2 * e] << 32 |
                                             (uint32_t)half_stage[16 + 2 * e]);
                q = A.cslot[at - f];
            }
        }
        if (q >= 0 && q != S.own) {
            EdmdPart r = A.p[q];
            double gr = G ? A.vr[q] : 0.0;
            if (SPEC && q == oth) {
                r.x = xo;
                r.y = yo;
                r.vx = vxo;
                r.vy = vyo;
                r.tl = t;
                r.coll = co;
                if (G) r.rad = ro;
            }
            if (W && !G && (C.field_on || C.damping)) {
                fly_v<true>(C, t, r.x, r.y, r.vx, r.vy, r.tl);
                if (!SPEC) {
                    /* a disk listed for both owners is written twice alike */
                    const auto w = A.p + q;
                    w->x = r.x;
                    w->y = r.y;
                    w->vx = r.vx;
                    w->vy = r.vy;
                    w->tl = r.tl;
                }
            }
            double tt;
            if (G)
                tt = coll_time_grow(C, t, S.x, S.y, S.vx, S.vy, S.r, S.vr, r.x, r.y, r.vx, r.vy,
                                    r.tl, r.rad, gr, S.ov);
            else
                tt = log_time<W>(C, coll_time_nb(C, t, S.x, S.y, S.vx, S.vy, S.r, r.x, r.y, r.vx,
                                                 r.vy, r.tl, r.rad, S.ov));
            if (tt < lim && tt < bt) {
                bt = tt;
                bq = q;
                bc = r.coll;
                bf = f;
            }
        }
    }
    WAVE_SYNC();
    double mt = half_min(bt);
    if (!two) {
        double a, b;
        halves(mt, a, b);
        mt = min_f64(a, b);
    }
    const uint64_t hit = __ballot(bt == mt);
    int wa = (int)__builtin_ctz((uint32_t)hit | (two ? 0u : 0x80000000u));
    int wb = 32 + (int)__builtin_ctz((uint32_t)(hit >> 32) | 0x80000000u);
    if (!two) wa = wb = (int)__builtin_ctzll(hit);
    if (passes > 1) {
        /* several passes: the lowest position among equal times */
        const uint64_t keep = two ? (hi ? hit >> 32 << 32 : (hit & 0xffffffffull)) : hit;
        if (__ballot(__popcll(keep) > 1)) {
            int fm = bt == mt ? bf : 0x7fffffff, l = lane;
            for (int m = 1; m < (two ? 32 : 64); m <<= 1) {
                const int of = __shfl_xor(fm, m, 64), ol = __shfl_xor(l, m, 64);
                if (of < fm) {
                    fm = of;
                    l = ol;
                }
            }
            wa = __builtin_amdgcn_readlane(l, 0);
            wb = __builtin_amdgcn_readlane(l, 32);
        }
    }
    const int w = 4 * (hi ? wb : wa);
    S.partner = __builtin_amdgcn_ds_bpermute(w, bq);
    S.cact = (uint32_t)__builtin_amdgcn_ds_bpermute(w, (int)bc);
    dt = mt;
    S.none0 = false;
    const bool none = !(mt < lim);
    if (__ballot(none)) {
        /* no candidate: partner 0 with its counter (EDMD.c:3091-3093), which
         * this event may have moved on */
        S.none0 = true;
        uint32_t c0 = A.p[0].coll;
        if (SPEC && S.kind != EVK_STALE && S.kind != EVK_CROSSING) {
            if (S.own == 0) c0 = S.coll;
            if (oth == 0) c0 = co;
        }
        if (none) {
            dt = lim;
            S.partner = 0;
            S.cact = c0;
        }
    }
}

/* The event's new collision and crossing times, absolute (SPEC as in
 * predict_halves). */
template <bool G, bool W, bool SPEC, class AR>
__device__ __forceinline__ void event_predict(const EdmdConst& C, const AR& A, int lane, double t,
                                              EvState& S, int32_t* stage) {
    double dt;
    predict_halves<G, W, SPEC>(C, A, lane, t, S, dt, stage);
    if (W && C.walls) {
        /* the wall time starts the reference's minimum: a neighbour
         * replaces it only when strictly earlier */
        const int typ = (C.walls & 8) ? A.ptype[S.own] : 0;
        double dw;
        int xy;
        const bool wall = G ? wall_time_grow(C, S.x, S.y, S.vx, S.vy, S.r, S.vr, S.cx, S.cy, dw,
                                             xy, typ)
                            : wall_time(C, S.x, S.y, S.vx, S.vy, S.r, S.cx, S.cy, dw, xy, typ);
        if (wall && !(dt < dw)) {
            dt = dw;
            S.partner = EDMD_WALL_CODE(xy);
            S.cact = 0;
        }
    }
    S.tk = t + dt;
    if (S.kind != EVK_STALE) {
        /* crossingEventGrow while growing: no field, no logTime */
        if (W && !G) cross_time<true>(C, t, S.x, S.y, S.vx, S.vy, S.cx, S.cy, S.tc, S.dir);
        else cross_rows(C, lane, t, S, S.tc, S.dir);
    }
}

/* The changed disks' records. */
template <class AR>
__device__ __forceinline__ void event_store(const AR& A, int lane, double t, const EvState& S) {
    if ((lane & 31) == 0 && (lane == 0 || S.nown == 2)) {
        EdmdPart r;
        r.x = S.x;
        r.y = S.y;
        r.vx = S.vx;
        r.vy = S.vy;
        r.tl = t;
        r.rad = S.r;
        r.m = S.m;
        r.coll = S.coll;
        r.cx = (int16_t)S.cx;
        r.cy = (int16_t)S.cy;
        A.p[S.own] = r;
    }
}

/* Insertions the event makes: crossings of i and j, then their collisions
 * (EDMD.c:3869-3879); a crossing or wall hit its crossing and collision
 * (EDMD.c:2587-2589, 3458-3459); a stale pop its collision. */
__device__ __forceinline__ int event_inserts(const EvState& S) {
    return S.kind == EVK_STALE ? 1 : 2 * S.nown;
}

/* Ranks of the event's new slots, filed with the queue at paulTime = paul
 * after ctr insertions, and its new leaves. */
__device__ __forceinline__ Leaf event_ranks(const EdmdConst& C, int lane, const EvState& S,
                                            double paul, int64_t ctr, int64_t& rk, int64_t& rx) {
    const bool stale = S.kind == EVK_STALE;
    const int64_t c = ctr + (lane >= 32 && S.nown == 2 ? 1 : 0);
    rx = stale ? S.rx_old : rank_of(S.tc, paul, C.dtp, C.horizon, c);
    rk = rank_of(S.tk, paul, C.dtp, C.horizon, c + (stale ? 0 : S.nown));
    return make_leaf(S.tk, rk, S.tc, rx, S.partner, S.dir);
}

/* The changed disks' slots, ranks and leaves, and a crossing's cell lists;
 * the records go by event_store. */
template <class AR>
__device__ __forceinline__ void event_slots(const AR& A, int lane, const EvState& S,
                                            const Leaf& L, int64_t rk, int64_t rx) {
    if ((lane & 31) == 0 && (lane == 0 || S.nown == 2)) {
        EdmdEv e;
        e.tcoll = S.tk;
        e.tcross = S.tc;
        e.partner = S.partner;
        e.cact = S.cact;
        e.dir = S.dir;
        e.pad = 0;
        A.e[S.own] = e;
        A.erank[2 * S.own] = rk;
        A.erank[2 * S.own + 1] = rx;
        EdmdNode n;
        n.key = L.key;
        n.idx = S.own;
        n.aux = L.aux;
        A.leaf[S.own] = n;
        A.lrank[S.own] = L.rank;
    }
}

/* Record k of the tape: a valid collision, or a hit of a flat wall (j = -1 -
 * xy, the normal and tangential velocities before the hit, resW, resT and
 * the contact coordinate). */
template <bool W, class AR>
__device__ __forceinline__ void tape_store(const EdmdConst& C, const AR& A, double t,
                                           const EvState& S, int p, int j, int64_t k) {
    if (k >= C.tape_cap) return;
    EdmdTapeRec rec;
    rec.t = t;
    rec.i = p;
    if (!W || S.kind == EVK_COLLISION) {
        rec.ax = S.dx;
        rec.ay = S.dy;
        rec.cx = S.dvx;
        rec.cy = S.dvy;
        rec.ff = S.ff;
        rec.j = j;
        rec.g = 0;
    } else {
        rec.ax = S.d == 0 ? S.vx0 : S.vy0;
        rec.ay = S.d == 0 ? S.vy0 : S.vx0;
        rec.cx = C.res_wall;
        rec.cy = C.res_tan;
        rec.ff = S.d == 0 ? S.x : S.y;
        rec.j = -1 - S.d;
        rec.g = C.field_on ? C.field : 0.0;
    }
    A.tape[k] = rec;
}

/* What a collision or a wall hit adds to the system's sums and its tape: the
 * collision virial (collTermX, collTermY, collTermXY, collTermYX) in vir, one
 * sum per lane, or the momentum given to the walls. */
template <bool G, bool W, class AR>
__device__ __forceinline__ void event_sums(const EdmdConst& C, const AR& A, int lane, double t,
                                           const EvState& S, int p, int j, double* vir) {
    if (G) return;
    EdmdState* st = A.st;
    const bool coll = !W || S.kind == EVK_COLLISION;
    if (coll && lane < 4) {
        const double u = (lane & 1) == 0 ? S.dx : S.dy;
        const double v = (lane == 0 || lane == 3) ? S.dx : S.dy;
        vir[lane] += S.w * u * v;
    }
    if (!coll && lane == 0) {
        st->dpw += S.dp;
        if (C.walls & 8) {
            st->dpl += S.dpl;
            st->dpm += S.dpm;
            st->dpr += S.dpr;
        }
    }
    if (C.tape_cap > 0 && lane == 0 && (coll || S.d != 2)) {
        const int64_t k = st->ntape;
        tape_store<W>(C, A, t, S, p, j, k);
        st->ntape = k + 1;
        if (coll) {
            st->wsum += S.w * (S.dx * S.dx + S.dy * S.dy);
            st->tlast = t;
        }
    }
}

/* removeFromCell and addToCell of a crossing: the cell left keeps the order
 * of the others; the new one gets p as its newest entry. */
template <class AR>
__device__ __forceinline__ void event_cells(const EdmdConst& C, const AR& A, int lane,
                                            const EvState& S) {
    const int p = S.own;
    const uint64_t hit = __ballot(lane < S.n0 && S.slot == p);
    const int pos = hit ? (int)__builtin_ctzll(hit) : S.n0;
    if (lane > pos && lane < S.n0) A.cslot[(size_t)S.c0 * C.cap + lane - 1] = S.slot;
    if (lane == 0) A.ccnt[S.c0] = S.n0 - 1;
    WAVE_SYNC();
}

template <class AR>
__device__ __forceinline__ void event_enter(const EdmdConst& C, const AR& A, int lane,
                                            const EvState& S, int n1) {
    if (lane == 0) {
        const int c1 = S.cy * C.ncx + S.cx;
        A.cslot[(size_t)c1 * C.cap + n1] = S.own; /* newest entry: visited first */
        A.ccnt[c1] = n1 + 1;
        const int wx = (S.d == 1 && S.cx == C.ncx - 1) ? -1 : ((S.d == 2 && S.cx == 0) ? 1 : 0);
        const int wy = (S.d == 3 && S.cy == C.ncy - 1) ? -1 : ((S.d == 4 && S.cy == 0) ? 1 : 0);
        if (wx) A.img[2 * S.own] += wx;
        if (wy) A.img[2 * S.own + 1] += wy;
    }
}

#endif
