/*
 * Prediction sweep kernels of libedmd_hip.so for gfx950.
 *
 *   k_sweep_tiled  prediction sweep: one workgroup per tile of cells (eight
 *                  tile shapes) stages the tile and its halo in LDS; one
 *                  lane per particle
 *                  computes the next cell crossing and the earliest
 *                  collision partner over the 3x3 cell neighbourhood
 *                  (EDMD.c:2405-2482, 2661-2723, 2829-3003; invoked for all
 *                  particles at EDMD.c:2007-2012 and 4909-4915)
 *   k_sweep_grow   the same for systems whose radii still grow
 *                  (collisionEventGrow, EDMD.c:3104-3230)
 *   k_sweep_count  counts a full sweep's insertions (the rank counter)
 *   k_tree_level   builds one level of the 64-ary minimum calendar
 *   k_sync_all     free flight of every particle to the system time
 *
 * Reference line numbers are those of src/EDMD.c.
 */
#define EDMD_DEVICE_ARRAYS 1
#include "edmd_device.h"

/* Cell-tiled sweep: one workgroup per SW_TX x SW_TY cells.  The tile and a
 * one-cell halo (wrapped periodically) are staged into LDS cell by cell in
 * row-major order, newest list entry first within a cell, so the three
 * cells of one row of a disk's 3x3 neighbourhood are one contiguous run
 * that lists the candidates in the reference's scan order (y offset outer,
 * x offset inner, newest entry first, EDMD.c:2959-3003).  Each thread
 * predicts one of the tile's disks over its three runs as one flat
 * candidate loop whose trip count is uniform over the wave; the loop keeps
 * only the cheap terms (approach b, contact d, discriminant) and marks the
 * candidates that can collide, and the roots of the marked ones are solved
 * afterwards in the same order with the strict-less rule, so the result is
 * that of predict_seq bit for bit.  Every disk record is read from HBM by
 * the one tile that owns it and the (at most eight) tiles whose halo holds
 * it, instead of once per neighbour scan that touches it.  Workgroups are
 * dealt to the eight XCDs round robin; tiles are renumbered so that each
 * XCD sweeps a contiguous band of tile rows and halo re-reads hit its own
 * L2.  A tile whose staged disks exceed SW_STAGE falls back to predict_seq
 * from global memory. */
/* Tile shapes of the sweep: TX x TY cells per workgroup of THREADS
 * threads; STAGE staged disks at most (tile plus halo). */
template <int TX_, int TY_, int THREADS_>
struct SweepShape {
    static constexpr int TX = TX_, TY = TY_, THREADS = THREADS_;
    static constexpr int HW = TX + 2, HH = TY + 2, NH = HW * HH;
    static constexpr int STAGE = 512;
    static_assert(NH <= 255, "staged cells carry a u8 index");
    static_assert(THREADS >= 64 && THREADS % 64 == 0, "whole waves");
};

/* The shapes a batch chooses from (edmd_batch_autotune times them; the
 * default is picked from the disks per cell).  At phi = 0.8 with unit
 * diameter a cell holds ~4.1 disks, at phi = 0.7 ~3.6, with the reference
 * CLI's radius 1 about one. */
using SweepV0 = SweepShape<8, 8, 320>;
using SweepV1 = SweepShape<6, 10, 256>;
using SweepV2 = SweepShape<10, 6, 256>;
using SweepV3 = SweepShape<8, 7, 256>;
using SweepV4 = SweepShape<8, 6, 192>;
using SweepV5 = SweepShape<8, 8, 256>;
using SweepV6 = SweepShape<8, 8, 64>;
using SweepV7 = SweepShape<16, 8, 128>;

/* The workgroup's LDS.  POLY = false is the layout of launches whose
 * systems all have equal radii: no radius per staged disk (4 KB less, one
 * more workgroup per CU).  The cell counts and the own-cell counts of the
 * two scans live in the velocity stage, which is written only after them. */
template <class S, bool POLY_>
struct SweepLds {
    static constexpr bool POLY = POLY_;
    /* staged disks: position flown to the sweep time, velocity, radius,
     * index, staged cell */
    double2 pos[S::STAGE], vel[S::STAGE];
    double rad[POLY ? S::STAGE : 1];
    int32_t id[S::STAGE];
    uint32_t coll[S::STAGE]; /* collision counter (the partner counter a prediction records) */
    uint8_t hcell[S::STAGE];
    int16_t own[S::STAGE];     /* staged index of each of the tile's own disks */
    int32_t start[S::NH + 1];  /* first staged index of each cell; [S::NH] = total */
    int32_t ostart[S::NH];     /* first own-list index of each tile cell */
    int32_t gcell[S::NH];
    int32_t ninner, total;
    static_assert(2 * S::NH * sizeof(int32_t) <= sizeof(vel), "scan counts fit the velocity stage");
    __device__ int32_t* cnt() { return reinterpret_cast<int32_t*>(&vel[0]); }
    __device__ int32_t* owncnt() { return reinterpret_cast<int32_t*>(&vel[0]) + S::NH; }
};

__device__ __forceinline__ int mod_cell(int a, int nc) {
    int r = a % nc;
    return r < 0 ? r + nc : r;
}

/* Exclusive scan of v over the NH staged cells by one wave (PER
 * consecutive cells per lane); returns the total.  Cells are ordered
 * h = (ly + 1) * HW + lx + 1. */
template <int NH>
__device__ __forceinline__ int sweep_scan(int lane, const int* v, int* out, int base) {
    constexpr int PER = (NH + 63) / 64;
    int val[PER];
    int sum = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int h = PER * lane + i;
        val[i] = h < NH ? v[h] : 0;
        sum += val[i];
    }
    int incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        int u = __shfl_up(incl, d, 64);
        if (lane >= d) incl += u;
    }
    int run = base + incl - sum;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int h = PER * lane + i;
        if (h < NH) out[h] = run;
        run += val[i];
    }
    return __shfl(incl, 63, 64);
}

/* The terms of collisionTime (EDMD.c:2661-2725) that decide whether a pair
 * can collide: relative position (minimum image when WRAP) and velocity,
 * approach b, |dv|^2, contact term d and discriminant, in the reference's
 * operation order. */
template <bool WRAP>
__device__ __forceinline__ void pair_terms(const EdmdConst& C, double ox, double oy, double ovx,
                                           double ovy, double orad, const double2 pv,
                                           const double2 vv, double r2, double& b, double& v2,
                                           double& d, double& det) {
    const double dvx = vv.x - ovx;
    const double dvy = vv.y - ovy;
    double dx = pv.x - ox;
    double dy = pv.y - oy;
    if (WRAP) min_image(C, dx, dy);
    b = dx * dvx + dy * dvy;
    v2 = dvx * dvx + dvy * dvy;
    d = dx * dx + dy * dy - 4 * orad * r2; /* DIST2, EDMD.c:35-43 */
    det = b * b - v2 * d;
}

/* The bits of the 64-bit mark word starting at candidate base that stay
 * set: candidates k < tot other than kself. */
__device__ __forceinline__ uint64_t keep_bits(int tot, int kself, int base) {
    return bits_below(tot - base) & ~bit_mask(kself - base);
}

/* The predictions of a staged tile's own disks, one thread per disk.  The
 * candidates of a disk are its three row runs, k = 0 .. tot-1 in scan
 * order.  Pass 1 runs k over the wave's largest tot (uniform) and marks in
 * a 256-bit mask the candidates with b <= 0 and det >= 0 (every other one
 * gives the reference's "never", which the strict-less minimum never
 * takes), flagging overlaps as collisionTime does; pass 2 solves the marked
 * roots in increasing k.  A disk with more than 256 candidates solves its
 * roots in pass 1 instead. */
template <class S, bool WRAP, bool X, bool MONO, class AR, class LD>
__device__ __forceinline__ void sweep_tile_predict(const EdmdConst& C, const AR& A, const LD& L,
                                                   int tid, int ninner, double t, int tx0, int ty0,
                                                   double paul, int64_t ctr0, double rad0,
                                                   bool& ov) {
    static_assert(MONO || LD::POLY, "unequal radii need the staged radii");
    const int lane = tid & 63;
    for (int u0 = tid - lane; u0 < ninner; u0 += S::THREADS) { /* uniform over the wave */
        const int u = u0 + lane;
        const bool act = u < ninner;
        const int me = L.own[act ? u : 0]; /* idle lanes shadow the first disk */
        const int h = L.hcell[me];
        const int lx = h % S::HW - 1, ly = h / S::HW - 1;
        /* the owner is synchronised at t (its staged position is its own) */
        const double2 opos = L.pos[me], ovel = L.vel[me];
        const double ox = opos.x, oy = opos.y, ovx = ovel.x, ovy = ovel.y;
        const double orad = LD::POLY ? L.rad[me] : rad0;
        const int p = L.id[me];
        /* row runs: cells (lx - 1 .. lx + 1, ly + j) are staged contiguously */
        const int h0 = ly * S::HW + lx;
        const int a0 = L.start[h0], n0 = L.start[h0 + 3] - a0;
        const int a1 = L.start[h0 + S::HW], n1 = L.start[h0 + S::HW + 3] - a1;
        const int a2 = L.start[h0 + 2 * S::HW], n2 = L.start[h0 + 2 * S::HW + 3] - a2;
        const int c1 = n0, c2 = n0 + n1;
        const int o0 = a0, o1 = a1 - c1, o2 = a2 - c2;
        const int tot = act ? c2 + n2 : 0;
        const bool direct = tot > 256;
        const int tot1 = direct ? 0 : tot;
        const int ktot = -wave_min_i32(-tot1);
        uint64_t m0 = 0, m1 = 0, m2 = 0, m3 = 0, cur = 0;
        double dt = EDMD_NEVER;
        int best = -1;
        int wxy = 2;
        bool wall = false;
        if (X && C.walls)
            wall = wall_time(C, ox, oy, ovx, ovy, orad, tx0 + lx, ty0 + ly, dt, wxy,
                             (C.walls & 8) ? A.ptype[p] : 0);
        /* pass 1 without branches: every lane evaluates its k-th candidate;
         * the marks of consecutive k collect in cur and go to their word
         * when k leaves it (k is uniform over the wave) */
        if constexpr (!WRAP) {
            /* The staged index advances by one per k and moves to the next
             * row run where that run starts; a lane past its own count reads
             * a staged disk clamped into the stage.  Only the discriminant
             * terms stay in the loop: the owner itself (k = kself) and the
             * k past the count are cleared from the marks afterwards, and
             * the overlap test moves to pass 2, since a pair with d < 0 and
             * b <= 0 always has det >= 0 and is marked. */
            int v = a0 - 1;
            uint32_t c32 = 0;
            for (int k = 0; k < ktot; ++k) {
                v = v + 1;
                v = k == c1 ? a1 : v;
                v = k == c2 ? a2 : v;
                const int vc = min(v, S::STAGE - 1);
                double b, v2, d, det;
                pair_terms<false>(C, ox, oy, ovx, ovy, orad, L.pos[vc], L.vel[vc],
                                  MONO ? orad : L.rad[vc], b, v2, d, det);
                if (!(b > 0) && !(det < 0)) c32 |= 1u << (k & 31);
                if ((k & 31) == 31 || k == ktot - 1) {
                    const uint64_t c = (k & 32) ? (uint64_t)c32 << 32 : (uint64_t)c32;
                    switch (k >> 6) {
                        case 0: m0 |= c; break;
                        case 1: m1 |= c; break;
                        case 2: m2 |= c; break;
                        default: m3 |= c; break;
                    }
                    c32 = 0;
                }
            }
            const int kself = c1 + (me - a1); /* the owner lies in its middle row run */
            m0 &= keep_bits(tot1, kself, 0);
            m1 &= keep_bits(tot1, kself, 64);
            m2 &= keep_bits(tot1, kself, 128);
            m3 &= keep_bits(tot1, kself, 192);
        } else
        for (int k = 0; k < ktot; ++k) {
            const bool in = k < tot1;
            const int vk = k + (k < c1 ? o0 : (k < c2 ? o1 : o2));
            const int v = in ? vk : me;
            double b, v2, d, det;
            pair_terms<WRAP>(C, ox, oy, ovx, ovy, orad, L.pos[v], L.vel[v],
                             MONO ? orad : L.rad[v], b, v2, d, det);
            /* the owner itself; a halo that wraps (boxes under three tiles
             * wide) may stage the owner's cell more than once */
            const bool self = WRAP ? L.id[v] == p : v == me;
            const bool ok = in && !self && !(b > 0);
            ov = ov || (ok && d < -0.01); /* EDMD.c:2708-2717 */
            const bool mark = ok && !(det < 0);
            cur |= mark ? ((uint64_t)1 << (k & 63)) : (uint64_t)0;
            if ((k & 63) == 63 || k == ktot - 1) {
                switch (k >> 6) {
                    case 0: m0 = cur; break;
                    case 1: m1 = cur; break;
                    case 2: m2 = cur; break;
                    default: m3 = cur; break;
                }
                cur = 0;
            }
        }
        /* disks with more than 256 candidates solve their roots in order as
         * they go */
        if (__ballot(direct)) {
            if (direct) {
                for (int k = 0; k < tot; ++k) {
                    const int v = k + (k < c1 ? o0 : (k < c2 ? o1 : o2));
                    if (WRAP ? L.id[v] == p : v == me) continue;
                    double b, v2, d, det;
                    pair_terms<WRAP>(C, ox, oy, ovx, ovy, orad, L.pos[v], L.vel[v],
                                     MONO ? orad : L.rad[v], b, v2, d, det);
                    if (b > 0) continue;
                    if (d < -0.01) ov = true;
                    if (det < 0) continue;
                    const double tt = log_time<X>(C, (-b - sqrt(det)) / v2);
                    if (dt > tt) {
                        dt = tt;
                        best = v;
                    }
                }
            }
        }
        /* the screen (uniform; not under damping, whose logTime could
         * merge distinct times): with q = -b > 0, the computed root
         * (q - fl(sqrt(det)))/v2 of a pair with d > 0 is at least
         * d/(2q) - 2^-25 q/v2 (its exact value lies in [d/(2q), d/q] and
         * the cancellation in det costs at most sqrt(3 2^-53) q/v2), so a
         * mark with d v2 - 2^-19 q^2 > 2 q v2 dt (1 + 2^-40) has a root
         * above the lane's best so far dt and is skipped: the strict-less
         * minimum never takes it (a skip needs d > 0, so d <= 0 pairs are
         * always solved) */
        const bool scr = C.screen != 0 && !(X && C.damping);
        uint32_t nmark = 0, nsolve = 0, nmiss = 0;
        while (m0 | m1 | m2 | m3) {
            int k;
            if (m0) { k = __builtin_ctzll(m0); m0 &= m0 - 1; }
            else if (m1) { k = 64 + __builtin_ctzll(m1); m1 &= m1 - 1; }
            else if (m2) { k = 128 + __builtin_ctzll(m2); m2 &= m2 - 1; }
            else { k = 192 + __builtin_ctzll(m3); m3 &= m3 - 1; }
            const int v = k + (k < c1 ? o0 : (k < c2 ? o1 : o2));
            double b, v2, d, det;
            pair_terms<WRAP>(C, ox, oy, ovx, ovy, orad, L.pos[v], L.vel[v],
                             MONO ? orad : L.rad[v], b, v2, d, det);
            if (!WRAP) ov = ov || d < -0.01; /* EDMD.c:2708-2717 */
            if (scr) {
                ++nmark;
                const double q = -b;
                const bool skip = dt > 0 && dt < EDMD_NEVER &&
                                  d * v2 - 0x1p-19 * (q * q) > (2 * q * v2 * dt) * (1 + 0x1p-40);
                if (skip) {
                    if (C.screen == 2 && !(log_time<X>(C, (-b - sqrt(det)) / v2) > dt)) ++nmiss;
                    continue;
                }
                ++nsolve;
            }
            const double tt = log_time<X>(C, (-b - sqrt(det)) / v2);
            if (dt > tt) {
                dt = tt;
                best = v;
            }
        }
        if (scr && C.screen == 2) { /* counted in the check mode only: the
                                       atomics contend on one address */
            uint32_t s0 = act ? nmark : 0, s1 = act ? nsolve : 0, s2 = act ? nmiss : 0;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                s0 += __shfl_xor(s0, off, 64);
                s1 += __shfl_xor(s1, off, 64);
                s2 += __shfl_xor(s2, off, 64);
            }
            if (lane == 0) {
                atomicAdd((unsigned long long*)&A.st->scr_marks, (unsigned long long)s0);
                atomicAdd((unsigned long long*)&A.st->scr_solved, (unsigned long long)s1);
                if (s2) atomicAdd((unsigned long long*)&A.st->scr_miss, (unsigned long long)s2);
            }
        }
        if (!act) continue;
        double tc;
        int dir;
        cross_time<X>(C, t, ox, oy, ovx, ovy, tx0 + lx, ty0 + ly, tc, dir);
        const double tk = t + dt;
        const int partner = best >= 0 ? L.id[best] : (wall ? EDMD_WALL_CODE(wxy) : 0);
        EdmdEv e;
        e.tcoll = tk;
        e.tcross = tc;
        e.partner = partner;
        /* the partner's counter from the stage; no partner: disk 0's
         * (EDMD.c:3091-3093 files partner 0) */
        e.cact = best >= 0 ? L.coll[best] : (partner >= 0 ? A.p[partner].coll : 0u);
        e.dir = dir;
        e.pad = 0;
        A.e[p] = e;
        const int64_t rk = rank_of(tk, paul, C.dtp, C.horizon, ctr0 + 2 * (int64_t)p + 1);
        const int64_t rx = rank_of(tc, paul, C.dtp, C.horizon, ctr0 + 2 * (int64_t)p);
        A.erank[2 * p] = rk;
        A.erank[2 * p + 1] = rx;
        const Leaf Lf = make_leaf(tk, rk, tc, rx, partner, dir);
        EdmdNode n;
        n.key = Lf.key;
        n.idx = p;
        n.aux = Lf.aux;
        A.leaf[p] = n;
        A.lrank[p] = Lf.rank;
    }
}

template <class S, bool X, bool POLY>
__global__ __launch_bounds__(S::THREADS) void k_sweep_tiled(const EdmdSys* __restrict__ systems) {
    __shared__ SweepLds<S, POLY> L;
    int32_t* const cnt = L.cnt();
    int32_t* const vtmp = L.owncnt();
    const EdmdSys* Sy = systems + blockIdx.y;
    const EdmdConst& C = Sy->c;
    const EdmdArrays& A = Sy->a;
    const int tid = threadIdx.x;
    if (A.st->growing) return; /* k_sweep_grow predicts growing systems */
    const int ncx = C.ncx, ncy = C.ncy;
    const int ntx = (ncx + S::TX - 1) / S::TX, nty = (ncy + S::TY - 1) / S::TY;
    const int per = gridDim.x / 8; /* gridDim.x is a multiple of 8 */
    const int tile = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
    if (tile >= ntx * nty) return; /* uniform over the workgroup */
    const int tx0 = (tile % ntx) * S::TX, ty0 = (tile / ntx) * S::TY;
    const int vw = min(S::TX, ncx - tx0), vh = min(S::TY, ncy - ty0);
    const double t = A.st->t;
    /* eventListInit order (EDMD.c:2007-2012): crossing then collision of
     * each particle in index order, after the insertions already counted */
    const double paul = A.st->paul;
    const int64_t ctr0 = A.st->ctr;

    for (int h = tid; h < S::NH; h += S::THREADS) {
        const int lx = h % S::HW - 1, ly = h / S::HW - 1;
        const int g = mod_cell(ty0 + ly, ncy) * ncx + mod_cell(tx0 + lx, ncx);
        L.gcell[h] = g;
        cnt[h] = A.ccnt[g];
    }
    __syncthreads();
    /* staged order: cells row-major (h), each cell newest entry first;
     * the tile's own cells also get consecutive places in the owner list */
    if (tid < 64) {
        constexpr int PER = (S::NH + 63) / 64;
        for (int h = PER * tid; h < PER * tid + PER && h < S::NH; ++h) {
            const int lx = h % S::HW - 1, ly = h / S::HW - 1;
            const bool own = lx >= 0 && lx < vw && ly >= 0 && ly < vh;
            vtmp[h] = own ? cnt[h] : 0;
        }
        const int nin = sweep_scan<S::NH>(tid, vtmp, L.ostart, 0);
        const int tot = sweep_scan<S::NH>(tid, cnt, L.start, 0);
        if (tid == 0) {
            L.start[S::NH] = tot;
            L.ninner = nin;
            L.total = tot;
        }
    }
    __syncthreads();
    const int total = L.total, ninner = L.ninner;
    bool ov = false;
    if (total <= S::STAGE) {
        const int cap = C.cap;
        for (int h = tid; h < S::NH; h += S::THREADS) {
            const int st0 = L.start[h], c = cnt[h];
            const int lx = h % S::HW - 1, ly = h / S::HW - 1;
            const bool own = lx >= 0 && lx < vw && ly >= 0 && ly < vh;
            for (int sl = 0; sl < c; ++sl) L.hcell[st0 + sl] = (uint8_t)h;
            if (own)
                for (int sl = 0; sl < c; ++sl) L.own[L.ostart[h] + sl] = (int16_t)(st0 + sl);
        }
        __syncthreads();
        /* two staged disks per thread and pass: both slot reads, then both
         * record reads, are in flight together; staged place st0 + i holds
         * list slot cnt - 1 - i */
        for (int u0 = tid; u0 < total; u0 += 2 * S::THREADS) {
            const int u1 = u0 + S::THREADS;
            const int h0 = L.hcell[u0];
            const int q0 = A.cslot[(size_t)L.gcell[h0] * cap + (L.start[h0 + 1] - 1 - u0)];
            int q1 = -1;
            if (u1 < total) {
                const int h1 = L.hcell[u1];
                q1 = A.cslot[(size_t)L.gcell[h1] * cap + (L.start[h1 + 1] - 1 - u1)];
            }
            const EdmdPart r0 = A.p[q0];
            EdmdPart r1;
            if (q1 >= 0) r1 = A.p[q1];
            const double lat0 = t - r0.tl;
            L.pos[u0] = make_double2(r0.x + lat0 * r0.vx, r0.y + lat0 * r0.vy);
            L.vel[u0] = make_double2(r0.vx, r0.vy);
            if (POLY) L.rad[u0] = r0.rad;
            L.id[u0] = q0;
            L.coll[u0] = r0.coll;
            if (q1 >= 0) {
                const double lat1 = t - r1.tl;
                L.pos[u1] = make_double2(r1.x + lat1 * r1.vx, r1.y + lat1 * r1.vy);
                L.vel[u1] = make_double2(r1.vx, r1.vy);
                if (POLY) L.rad[u1] = r1.rad;
                L.id[u1] = q1;
                L.coll[u1] = r1.coll;
            }
        }
        __syncthreads();
        /* a tile whose halo stays off the seam, in a box at least five
         * cells wide: every candidate lies within two cells of its owner,
         * so the minimum image (EDMD.c:5896-5913) changes nothing and is
         * skipped (uniform over the workgroup).  The last cell column and
         * row are seam cells: a leftward (downward) crossing out of cell 0
         * can leave x (y) at +0 there (PBCpostX wraps only x < 0,
         * EDMD.c:5948-5953), and a disk with t_local = t keeps it when
         * synchronised, so a halo holding them needs the minimum image.
         * Column and row 0 are only ever halo of tiles that wrap. */
        const bool nowrap = tx0 >= 1 && ty0 >= 1 && tx0 + vw <= ncx - 2 && ty0 + vh <= ncy - 2 &&
                            ncx >= 5 && ncy >= 5;
        /* equal radii: the contact term 4 r r of every pair is the owner's
         * own (bitwise the same product), no radius read per candidate;
         * without staged radii it is disk 0's (every radius is bitwise the
         * same) */
        const double rad0 = POLY ? 0.0 : A.p[0].rad;
        if constexpr (!POLY) {
            if (nowrap)
                sweep_tile_predict<S, false, X, true>(C, A, L, tid, ninner, t, tx0, ty0, paul, ctr0,
                                                      rad0, ov);
            else
                sweep_tile_predict<S, true, X, true>(C, A, L, tid, ninner, t, tx0, ty0, paul, ctr0,
                                                     rad0, ov);
        } else {
            if (nowrap && C.mono)
                sweep_tile_predict<S, false, X, true>(C, A, L, tid, ninner, t, tx0, ty0, paul, ctr0,
                                                      rad0, ov);
            else if (nowrap)
                sweep_tile_predict<S, false, X, false>(C, A, L, tid, ninner, t, tx0, ty0, paul,
                                                       ctr0, rad0, ov);
            else
                sweep_tile_predict<S, true, X, false>(C, A, L, tid, ninner, t, tx0, ty0, paul, ctr0,
                                                      rad0, ov);
        }
    } else {
        const int cap = C.cap;
        for (int w = tid; w < S::TX * S::TY * cap; w += S::THREADS) {
            const int c = w / cap, sl = w - c * cap;
            const int lx = c % S::TX, ly = c / S::TX;
            if (lx >= vw || ly >= vh) continue;
            const int g = (ty0 + ly) * ncx + tx0 + lx;
            if (sl < A.ccnt[g]) {
                const int q = A.cslot[(size_t)g * cap + sl];
                ov |= sweep_one<false, X>(C, A, t, q, paul, ctr0 + 2 * (int64_t)q,
                                       ctr0 + 2 * (int64_t)q + 1);
            }
        }
    }
    if (ov) atomicExch(&A.st->status, EDMD_DEV_OVERLAP);
}

__global__ __launch_bounds__(256) void k_tree_level(const EdmdSys* __restrict__ systems, int l) {
    const EdmdSys* S = systems + blockIdx.y;
    if (l > S->c.nlev) return;
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= S->c.lsize[l]) return;
    node_min(S->c, S->a, l, g);
}

__global__ __launch_bounds__(256) void k_sync_all(const EdmdSys* __restrict__ systems) {
    const EdmdSys* S = systems + blockIdx.y;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= S->c.n) return;
    const double t = S->a.st->t;
    EdmdPart* r = S->a.p + p;
    double x = r->x, y = r->y, tl = r->tl;
    if (S->a.st->growing) {
        double rad = r->rad;
        fly_grow(S->c, t, x, y, r->vx, r->vy, tl, rad, S->a.vr[p]);
        r->rad = rad;
    } else {
        double vx = r->vx, vy = r->vy;
        fly_v<true>(S->c, t, x, y, vx, vy, tl);
        r->vx = vx;
        r->vy = vy;
    }
    r->x = x;
    r->y = y;
    r->tl = tl;
}

/* Prediction sweep of the systems that are growing (collisionEventGrow,
 * EDMD.c:3104-3230, crossingEventGrow, EDMD.c:2343-2400 = the Normal
 * crossing), one lane per particle. */
__global__ __launch_bounds__(256) void k_sweep_grow(const EdmdSys* __restrict__ systems) {
    const EdmdSys* S = systems + blockIdx.y;
    if (!S->a.st->growing) return;
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= S->c.n) return;
    const int64_t ctr0 = S->a.st->ctr;
    bool ov = sweep_one<true>(S->c, S->a, S->a.st->t, p, S->a.st->paul, ctr0 + 2 * (int64_t)p,
                              ctr0 + 2 * (int64_t)p + 1);
    if (ov) atomicExch(&S->a.st->status, EDMD_DEV_OVERLAP);
}

/* After a full sweep: one insertion per slot of every particle counted. */
__global__ void k_sweep_count(const EdmdSys* __restrict__ systems, int nsys) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < nsys) systems[s].a.st->ctr += 2 * (int64_t)systems[s].c.n;
}

/* ------------------------------------------------------------ launchers */

template <class S>
static void launch_sweep(const EdmdSys* d_sys, int nsys, int max_tiles, int ext, hipStream_t s) {
    dim3 grid((max_tiles + 7) / 8 * 8, nsys);
    if (ext & EDMD_SWEEP_EXT)
        hipLaunchKernelGGL((k_sweep_tiled<S, true, true>), grid, dim3(S::THREADS), 0, s, d_sys);
    else if (ext & EDMD_SWEEP_POLY)
        hipLaunchKernelGGL((k_sweep_tiled<S, false, true>), grid, dim3(S::THREADS), 0, s, d_sys);
    else
        hipLaunchKernelGGL((k_sweep_tiled<S, false, false>), grid, dim3(S::THREADS), 0, s, d_sys);
}

hipError_t edmd_launch_sweep_tiled(const EdmdSys* d_sys, int nsys, int max_tiles, int variant,
                                   int ext, hipStream_t s) {
    if (nsys <= 0 || max_tiles <= 0) return hipSuccess;
    switch (variant) {
        case 0: launch_sweep<SweepV0>(d_sys, nsys, max_tiles, ext, s); break;
        case 1: launch_sweep<SweepV1>(d_sys, nsys, max_tiles, ext, s); break;
        case 2: launch_sweep<SweepV2>(d_sys, nsys, max_tiles, ext, s); break;
        case 3: launch_sweep<SweepV3>(d_sys, nsys, max_tiles, ext, s); break;
        case 4: launch_sweep<SweepV4>(d_sys, nsys, max_tiles, ext, s); break;
        case 5: launch_sweep<SweepV5>(d_sys, nsys, max_tiles, ext, s); break;
        case 6: launch_sweep<SweepV6>(d_sys, nsys, max_tiles, ext, s); break;
        case 7: launch_sweep<SweepV7>(d_sys, nsys, max_tiles, ext, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <class S>
static EdmdSweepShape shape_of() {
    return EdmdSweepShape{S::TX, S::TY, S::THREADS, S::STAGE};
}

EdmdSweepShape edmd_sweep_shape(int variant) {
    switch (variant) {
        case 0: return shape_of<SweepV0>();
        case 1: return shape_of<SweepV1>();
        case 2: return shape_of<SweepV2>();
        case 3: return shape_of<SweepV3>();
        case 4: return shape_of<SweepV4>();
        case 5: return shape_of<SweepV5>();
        case 6: return shape_of<SweepV6>();
        case 7: return shape_of<SweepV7>();
        default: return EdmdSweepShape{0, 0, 0, 0};
    }
}

int edmd_sweep_tiles(int ncx, int ncy, int variant) {
    const EdmdSweepShape sh = edmd_sweep_shape(variant);
    if (sh.tx <= 0) return 0;
    return ((ncx + sh.tx - 1) / sh.tx) * ((ncy + sh.ty - 1) / sh.ty);
}

hipError_t edmd_launch_tree(const EdmdSys* d_sys, int nsys, const int* max_lsize, int max_nlev,
                            hipStream_t s) {
    for (int l = 1; l <= max_nlev; ++l) {
        dim3 grid((max_lsize[l] + 255) / 256, nsys);
        hipLaunchKernelGGL(k_tree_level, grid, dim3(256), 0, s, d_sys, l);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t edmd_launch_sync_all(const EdmdSys* d_sys, int nsys, int max_n, hipStream_t s) {
    dim3 grid((max_n + 255) / 256, nsys);
    hipLaunchKernelGGL(k_sync_all, grid, dim3(256), 0, s, d_sys);
    return hipGetLastError();
}

hipError_t edmd_launch_sweep_grow(const EdmdSys* d_sys, int nsys, int max_n, hipStream_t s) {
    if (nsys <= 0 || max_n <= 0) return hipSuccess;
    dim3 grid((max_n + 255) / 256, nsys);
    hipLaunchKernelGGL(k_sweep_grow, grid, dim3(256), 0, s, d_sys);
    return hipGetLastError();
}

hipError_t edmd_launch_sweep_count(const EdmdSys* d_sys, int nsys, hipStream_t s) {
    hipLaunchKernelGGL(k_sweep_count, dim3((nsys + 255) / 256), dim3(256), 0, s, d_sys, nsys);
    return hipGetLastError();
}
