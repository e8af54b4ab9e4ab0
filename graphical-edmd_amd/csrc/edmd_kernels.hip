/*
 * Single-step and utility kernels of libedmd_hip.so for gfx950 (CDNA4,
 * 64-lane wavefronts).
 *
 *   k_epoch_begin, k_epoch_end
 *                  per-system bounds and counters of graph-captured epochs
 *   k_peek, k_pair_time, k_repredict, k_queue_edit, k_fly_one
 *                  single steps for the reference-compatible entry points
 *   k_pcf          g(r) (pcf.c:16-75) of all pairs, without scratch memory
 *   k_fp64_check   IEEE division / square root probe for the tests
 *
 * Reference line numbers are those of src/EDMD.c.
 */
#define EDMD_DEVICE_ARRAYS 1
#include "edmd_loop.h"
#include "edmd_variants.h"

/* ------------------------------------------------------------ single steps */

/* findNextEvent, EDMD.c:2313-2327: the earliest pending event, particle or
 * scheduled, without handling it. */
__global__ __launch_bounds__(64) void k_peek(const EdmdSys* __restrict__ systems, EdmdPeek* out) {
    const EdmdConst& C = systems[blockIdx.x].c;
    const EdmdArrays& A = systems[blockIdx.x].a;
    const int lane = threadIdx.x;
    double key;
    int p, aux;
    top_min(C, A, lane, level(A, C.nlev), A.st->t, key, p, aux);
    __shared__ QueueState Qs;
    LoopRegs R;
    R.q = &Qs;
    next_special(A.st, R);
    const int64_t krank = key == R.next_special ? uni64(A.lrank[p]) : (int64_t)0;
    if (lane != 0) return;
    EdmdPeek r;
    if (!before(key, krank, R.next_special, R.srank)) {
        r.t = R.next_special; r.type = R.special; r.i = 0; r.j = 0; r.coll_actual = 0;
    } else if (aux >= 0) {
        r.t = key; r.type = EDMD_EV_COLLISION; r.i = p; r.j = aux; r.coll_actual = A.e[p].cact;
    } else if (aux <= EDMD_WALL_CODE(0)) {
        r.t = key; r.type = EDMD_EV_WALL; r.i = p; r.j = EDMD_WALL_CODE(0) - aux; r.coll_actual = 0;
    } else {
        r.t = key; r.type = EDMD_EV_CELLCROSS; r.i = p; r.j = -aux; r.coll_actual = 0;
    }
    out[blockIdx.x] = r;
}

/* collisionTimeNormal(p1, p2) at the system time, EDMD.c:2661-2723; p1 is
 * taken at its stored position as the reference does. */
__global__ void k_pair_time(const EdmdSys* __restrict__ systems, int i, int j, double* out) {
    const EdmdConst& C = systems[0].c;
    const EdmdArrays& A = systems[0].a;
    bool ov = false;
    const double t = A.st->t;
    const EdmdPart a = A.p[i], b = A.p[j];
    if (A.st->growing)
        out[0] = coll_time_grow(C, t, a.x, a.y, a.vx, a.vy, a.rad, A.vr[i], b.x, b.y, b.vx, b.vy,
                                b.tl, b.rad, A.vr[j], ov);
    else
        out[0] = coll_time(C, t, a.x, a.y, a.vx, a.vy, a.rad, b.x, b.y, b.vx, b.vy, b.tl, b.rad, ov);
    out[1] = ov ? 1.0 : 0.0;
}

/* collisionEvent(i) / crossingEvent(i) for one particle (which: bit 0 =
 * crossing, bit 1 = collision) at the system time, then the calendar path
 * of i is updated. */
template <int ML>
__global__ __launch_bounds__(64) void k_repredict(const EdmdSys* __restrict__ systems, int i,
                                                 int which) {
    const EdmdConst& C = systems[0].c;
    const EdmdArrays& A = systems[0].a;
    const int lane = threadIdx.x;
    __shared__ int32_t stage[EDMD_STAGE_MAX];
    const double t = A.st->t;
    const EdmdPart pi = A.p[i];
    EdmdEv e = A.e[i];
    PathCache<ML> P;
    path_prefetch<ML>(C, A, lane, i, -1, P);
    const double paul = A.st->paul;
    int64_t ctr = A.st->ctr;
    int64_t rcoll = A.erank[2 * i], rcross = A.erank[2 * i + 1];
    if (which & 1) {
        cross_time(C, t, pi.x, pi.y, pi.vx, pi.vy, pi.cx, pi.cy, e.tcross, e.dir);
        rcross = rank_of(e.tcross, paul, C.dtp, C.horizon, ctr++);
    }
    bool ov = false;
    if (which & 2) {
        const bool grow = uni(A.st->growing) != 0;
        EvState S;
        S.own = i;
        S.x = pi.x; S.y = pi.y; S.vx = pi.vx; S.vy = pi.vy; S.r = pi.rad; S.m = pi.m;
        S.vr = grow ? A.vr[i] : 0.0;
        S.coll = pi.coll; S.cx = pi.cx; S.cy = pi.cy;
        S.kind = EVK_STALE; /* the collision slot alone */
        S.nown = 1;
        S.ov = false;
        if (grow) event_predict<true, true, false>(C, A, lane, t, S, stage);
        else event_predict<false, true, false>(C, A, lane, t, S, stage);
        ov = S.ov;
        e.partner = S.partner;
        e.cact = S.cact;
        e.tcoll = S.tk;
        rcoll = rank_of(e.tcoll, paul, C.dtp, C.horizon, ctr++);
    }
    if (lane == 0) {
        A.e[i] = e;
        A.erank[2 * i] = rcoll;
        A.erank[2 * i + 1] = rcross;
    }
    const Leaf L = make_leaf(e.tcoll, rcoll, e.tcross, rcross, e.partner, e.dir);
    leaf_store(A, lane, i, L);
    path_update<ML>(C, A, lane, P, i, L.key, L.aux, -1, 0.0, 0, nullptr, t);
    const bool any_ov = __ballot(ov) != 0ull;
    if (lane == 0) {
        A.st->ctr = ctr;
        if (any_ov) {
            A.st->status = EDMD_DEV_OVERLAP;
            A.st->err_i = i;
        }
    }
}

/* addEventToQueue / removeEventFromQueue (EDMD.c:2144-2221) on one slot of
 * the reference's eventList, as a caller fills it (addCollisionEvent,
 * addCrossingEvent, addWallEvent, addEvent*: EDMD.c:2487-2496, 3286-3297,
 * 3321-3330, 4421-4440, 4814-4822).  mode 0: file the slot at time t with
 * partner / direction / wall side j and partner counter cact; mode 1: the
 * same with the partner's current counter (addCollisionEvent); mode 2:
 * take the slot out (it never pops until filed again).  A filed slot takes
 * the next insertion rank, as the reference's queue orders it. */
template <int ML>
__global__ __launch_bounds__(64) void k_queue_edit(const EdmdSys* __restrict__ systems, int kind,
                                                  int i, int j, double t, uint32_t cact,
                                                  int mode) {
    const EdmdConst& C = systems[0].c;
    const EdmdArrays& A = systems[0].a;
    const int lane = threadIdx.x;
    EdmdState* st = A.st;
    const double paul = st->paul;
    int64_t ctr = st->ctr;
    const bool remove = mode == 2;
    if (kind == EDMD_EV_SCREENSHOT || kind == EDMD_EV_THERMO || kind == EDMD_EV_ADDINGNOISE) {
        const double tn = remove ? INF_D : t;
        const int64_t rk = remove ? INT64_MAX : rank_of(t, paul, C.dtp, C.horizon, ctr);
        const int64_t wk = remove ? INT64_MAX : window_of(t, paul, C.dtp, C.nlists, st->win);
        if (!remove) ctr++;
        if (lane == 0) {
            if (kind == EDMD_EV_SCREENSHOT) {
                st->next_screen = tn; st->rank_screen = rk; st->win_screen = wk;
            } else if (kind == EDMD_EV_THERMO) {
                st->next_thermo = tn; st->rank_thermo = rk; st->win_thermo = wk;
            } else {
                st->next_noise = tn; st->rank_noise = rk; st->win_noise = wk;
            }
            st->ctr = ctr;
        }
        return;
    }
    EdmdEv e = A.e[i];
    int64_t rcoll = A.erank[2 * i], rcross = A.erank[2 * i + 1];
    PathCache<ML> P;
    path_prefetch<ML>(C, A, lane, i, -1, P);
    if (kind == EDMD_EV_CELLCROSS) {
        if (remove) {
            e.tcross = INF_D;
        } else {
            e.tcross = t;
            e.dir = j;
            rcross = rank_of(t, paul, C.dtp, C.horizon, ctr++);
        }
    } else {
        if (remove) {
            e.tcoll = INF_D;
        } else {
            e.tcoll = t;
            e.partner = kind == EDMD_EV_WALL ? EDMD_WALL_CODE(j) : j;
            e.cact = kind == EDMD_EV_WALL ? 0u : (mode == 1 ? A.p[j].coll : cact);
            rcoll = rank_of(t, paul, C.dtp, C.horizon, ctr++);
        }
    }
    if (lane == 0) {
        A.e[i] = e;
        A.erank[2 * i] = rcoll;
        A.erank[2 * i + 1] = rcross;
    }
    const Leaf L = make_leaf(e.tcoll, rcoll, e.tcross, rcross, e.partner, e.dir);
    leaf_store(A, lane, i, L);
    path_update<ML>(C, A, lane, P, i, L.key, L.aux, -1, 0.0, 0, nullptr, st->t);
    if (lane == 0) st->ctr = ctr;
}

/* freeFlyNormal(p) at the system time, EDMD.c:4954-4990. */
__global__ void k_fly_one(const EdmdSys* __restrict__ systems, int i) {
    const EdmdConst& C = systems[0].c;
    const EdmdArrays& A = systems[0].a;
    EdmdPart* r = A.p + i;
    double x = r->x, y = r->y, tl = r->tl;
    if (A.st->growing) {
        double rad = r->rad;
        fly_grow(C, A.st->t, x, y, r->vx, r->vy, tl, rad, A.vr[i]);
        r->rad = rad;
    } else {
        double vx = r->vx, vy = r->vy;
        fly_v<true>(C, A.st->t, x, y, vx, vy, tl);
        r->vx = vx;
        r->vy = vy;
    }
    r->x = x;
    r->y = y;
    r->tl = tl;
}

/* calculate_pcf, pcf.c:16-75: histogram of minimum-image pair distances
 * below rmax = dr * nb, one count per unordered pair (the reference adds
 * 2.0 per pair; the host doubles the counts).  Blocks take 256 x 256 tiles
 * of the upper pair triangle and count into an LDS histogram.  For callers
 * without scratch memory; k_pcf_pairs has the others.  extrap != 0
 * uses positions free-flown to time t without storing them. */
__global__ __launch_bounds__(256) void k_pcf(const double* __restrict__ px,
                                            const double* __restrict__ py,
                                            const EdmdPart* __restrict__ part, int n, double t,
                                            int extrap, double Lx, double Ly, double dr, int nb,
                                            unsigned long long* __restrict__ hist) {
    extern __shared__ unsigned int h[];
    __shared__ double sx[256], sy[256];
    const int ti = blockIdx.x, tj = blockIdx.y;
    if (tj < ti) return;
    const double halfLx = Lx / 2, halfLy = Ly / 2;
    const double rmax = dr * nb;
    for (int b = threadIdx.x; b < nb; b += 256) h[b] = 0;
    auto pos = [&](int q, double& xx, double& yy) {
        if (part) {
            const EdmdPart r = part[q];
            xx = r.x;
            yy = r.y;
            if (extrap) {
                double dt = t - r.tl;
                xx += dt * r.vx;
                yy += dt * r.vy;
                xx = wrap_post(xx, Lx);
                yy = wrap_post(yy, Ly);
            }
        } else {
            xx = px[q];
            yy = py[q];
        }
    };
    const int j0 = tj * 256;
    if (j0 + (int)threadIdx.x < n) pos(j0 + threadIdx.x, sx[threadIdx.x], sy[threadIdx.x]);
    __syncthreads();
    const int i = ti * 256 + threadIdx.x;
    if (i < n) {
        double xi, yi;
        pos(i, xi, yi);
        const int jn = min(256, n - j0);
        for (int k = 0; k < jn; ++k) {
            const int j = j0 + k;
            if (j <= i) continue;
            double dx = sx[k] - xi;
            double dy = sy[k] - yi;
            if (dx >= halfLx) dx -= Lx;
            else if (dx < -halfLx) dx += Lx;
            if (dy >= halfLy) dy -= Ly;
            else if (dy < -halfLy) dy += Ly;
            double r = sqrt(dx * dx + dy * dy);
            if (r < rmax) {
                int bin = (int)(r / dr);
                if (bin < nb) atomicAdd(&h[bin], 1u);
            }
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nb; b += 256)
        if (h[b]) atomicAdd(&hist[b], (unsigned long long)h[b]);
}

__global__ void k_fp64_check(int n, const double* __restrict__ a, const double* __restrict__ b,
                             double* __restrict__ q, double* __restrict__ s) {
    int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    q[k] = a[k] / b[k];
    s[k] = sqrt(a[k]);
}

/* Members of rows as arrays, a row a thread, into pinned host memory: the
 * host copies whole arrays where it picked each member out of 64-byte rows,
 * eight passes over lines that the card had just written (the state of 300000
 * disks 1046 us to 734).  The stores are whole lines; the rows' lines come
 * from the caches after their first member. */
__global__ __launch_bounds__(256) void k_columns(const unsigned char* __restrict__ rows, int64_t n,
                                                 unsigned char* __restrict__ out, EdmdColumns cols) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const unsigned char* const r = rows + i * cols.row;
#pragma unroll
    for (int c = 0; c < EDMD_COLUMNS; ++c) {
        if (c >= cols.n) break;
        const unsigned char* const at = r + cols.src[c];
        unsigned char* const to = out + cols.dst[c];
        if (cols.kind[c] == 8) ((double*)to)[i] = *(const double*)at;
        else if (cols.kind[c] == 4) ((int32_t*)to)[i] = *(const int32_t*)at;
        else ((int32_t*)to)[i] = *(const int16_t*)at;
    }
}

/* ------------------------------------------------------------ launchers */

/* Epochs of a graph-captured run: the bounds of the coming epoch relative
 * to each system's counters (one thread per system), and each system's
 * counters when the epoch has run. */
__global__ __launch_bounds__(256) void k_epoch_begin(const EdmdSys* __restrict__ systems, int nsys,
                                                     int64_t ev_inc, uint64_t coll_inc) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsys) return;
    EdmdState EDMD_GLOBAL* st = systems[s].a.st;
    const uint64_t ne = st->nevents, nc = st->ncol;
    st->ev_limit = ev_inc > INT64_MAX - (int64_t)ne ? INT64_MAX : (int64_t)ne + ev_inc;
    st->coll_limit = coll_inc > ~(uint64_t)0 - nc ? ~(uint64_t)0 : nc + coll_inc;
}

__global__ __launch_bounds__(256) void k_epoch_end(const EdmdSys* __restrict__ systems, int nsys,
                                                   EdmdEpochRow* __restrict__ rows) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nsys) return;
    const EdmdState EDMD_GLOBAL* st = systems[s].a.st;
    EdmdEpochRow r;
    r.t = st->t;
    r.ncol = st->ncol;
    r.ncross = st->ncross;
    r.nevents = st->nevents;
    r.status = st->status;
    r.stop_reason = st->stop_reason;
    rows[s] = r;
}

hipError_t edmd_launch_epoch_begin(const EdmdSys* d_sys, int nsys, int64_t ev_inc,
                                   uint64_t coll_inc, hipStream_t s) {
    hipLaunchKernelGGL(k_epoch_begin, dim3((nsys + 255) / 256), dim3(256), 0, s, d_sys, nsys,
                       ev_inc, coll_inc);
    return hipGetLastError();
}

hipError_t edmd_launch_epoch_end(const EdmdSys* d_sys, int nsys, EdmdEpochRow* rows,
                                 hipStream_t s) {
    hipLaunchKernelGGL(k_epoch_end, dim3((nsys + 255) / 256), dim3(256), 0, s, d_sys, nsys, rows);
    return hipGetLastError();
}

hipError_t edmd_launch_run(const EdmdSys* d_sys, int nsys, int max_nlev, int grow, int walls,
                           int wpb, EdmdRunArgs ra, hipStream_t s) {
    if (wpb != 1 && (grow || walls || max_nlev > 2 || (wpb != 2 && wpb != 4)))
        return hipErrorInvalidValue;
    if (wpb != 1) EdmdLoopVariant<false, false>::run_packed(d_sys, nsys, max_nlev, wpb, ra, s);
    else if (grow && walls) EdmdLoopVariant<true, true>::run(d_sys, nsys, max_nlev, ra, s);
    else if (grow) EdmdLoopVariant<true, false>::run(d_sys, nsys, max_nlev, ra, s);
    else if (walls) EdmdLoopVariant<false, true>::run(d_sys, nsys, max_nlev, ra, s);
    else EdmdLoopVariant<false, false>::run(d_sys, nsys, max_nlev, ra, s);
    return hipGetLastError();
}

static const void* lds_kernel(int max_nlev, int grow, int walls) {
    if (grow)
        return walls ? EdmdLoopVariant<true, true>::lds_kernel(max_nlev)
                     : EdmdLoopVariant<true, false>::lds_kernel(max_nlev);
    return walls ? EdmdLoopVariant<false, true>::lds_kernel(max_nlev)
                 : EdmdLoopVariant<false, false>::lds_kernel(max_nlev);
}

hipError_t edmd_lds_occupancy(int max_nlev, int grow, int walls, size_t dyn_bytes,
                              int* blocks_per_cu, size_t* static_bytes) {
    const void* f = lds_kernel(max_nlev, grow, walls);
    *blocks_per_cu = 0;
    *static_bytes = 0;
    if (!f) return hipErrorInvalidValue;
    hipFuncAttributes fa;
    hipError_t e = hipFuncGetAttributes(&fa, f);
    if (e != hipSuccess) return e;
    *static_bytes = fa.sharedSizeBytes;
    e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)dyn_bytes);
    if (e != hipSuccess) return e;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, f, 64, dyn_bytes);
}

hipError_t edmd_launch_run_lds(const EdmdSys* d_sys, int nsys, int max_nlev, int grow, int walls,
                               size_t dyn_bytes, EdmdRunArgs ra, hipStream_t s) {
    if (max_nlev > 2) return hipErrorInvalidValue;
    if (grow && walls) EdmdLoopVariant<true, true>::run_lds(d_sys, nsys, max_nlev, dyn_bytes, ra, s);
    else if (grow) EdmdLoopVariant<true, false>::run_lds(d_sys, nsys, max_nlev, dyn_bytes, ra, s);
    else if (walls) EdmdLoopVariant<false, true>::run_lds(d_sys, nsys, max_nlev, dyn_bytes, ra, s);
    else EdmdLoopVariant<false, false>::run_lds(d_sys, nsys, max_nlev, dyn_bytes, ra, s);
    return hipGetLastError();
}

static const void* wide_kernel(int grow, int walls, int waves, int place) {
    if (grow)
        return walls ? EdmdWideVariant<true, true>::kernel(waves, place)
                     : EdmdWideVariant<true, false>::kernel(waves, place);
    return walls ? EdmdWideVariant<false, true>::kernel(waves, place)
                 : EdmdWideVariant<false, false>::kernel(waves, place);
}

hipError_t edmd_wide_occupancy(int grow, int walls, int waves, int place, size_t dyn_bytes,
                               int* blocks_per_cu) {
    *blocks_per_cu = 0;
    const void* f = wide_kernel(grow, walls, waves, place);
    if (!f) return hipErrorInvalidValue;
    int dev = 0, maxblk = 0;
    hipFuncAttributes fa;
    hipError_t e = hipFuncGetAttributes(&fa, f);
    if (e == hipSuccess) e = hipGetDevice(&dev);
    if (e == hipSuccess)
        e = hipDeviceGetAttribute(&maxblk, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (e != hipSuccess) return e;
    if (fa.sharedSizeBytes + dyn_bytes > (size_t)maxblk) return hipSuccess; /* none fits */
    /* the kernel's own limit, the same whatever the batch */
    e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                            maxblk - (int)fa.sharedSizeBytes);
    if (e != hipSuccess) return e;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, f, 64 * waves, dyn_bytes);
}

hipError_t edmd_launch_run_wide(const EdmdSys* d_sys, int nsys, int grow, int walls, int waves,
                                int place, size_t dyn_bytes, EdmdRunArgs ra, hipStream_t s) {
    if (grow && walls) return EdmdWideVariant<true, true>::run(waves, place, d_sys, nsys, dyn_bytes, ra, s);
    if (grow) return EdmdWideVariant<true, false>::run(waves, place, d_sys, nsys, dyn_bytes, ra, s);
    if (walls) return EdmdWideVariant<false, true>::run(waves, place, d_sys, nsys, dyn_bytes, ra, s);
    return EdmdWideVariant<false, false>::run(waves, place, d_sys, nsys, dyn_bytes, ra, s);
}

hipError_t edmd_launch_columns(const void* rows, int64_t n, void* out, const EdmdColumns& cols,
                               hipStream_t s) {
    if (n < 1 || cols.n < 1) return hipSuccess;
    hipLaunchKernelGGL(k_columns, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                       (const unsigned char*)rows, n, (unsigned char*)out, cols);
    return hipGetLastError();
}

hipError_t edmd_launch_peek(const EdmdSys* d_sys, int nsys, EdmdPeek* out, hipStream_t s) {
    hipLaunchKernelGGL(k_peek, dim3(nsys), dim3(64), 0, s, d_sys, out);
    return hipGetLastError();
}

hipError_t edmd_launch_pair_time(const EdmdSys* d_sys, int i, int j, double* out, hipStream_t s) {
    hipLaunchKernelGGL(k_pair_time, dim3(1), dim3(1), 0, s, d_sys, i, j, out);
    return hipGetLastError();
}

hipError_t edmd_launch_repredict(const EdmdSys* d_sys, int max_nlev, int i, int which,
                                 hipStream_t s) {
    if (max_nlev <= 1) hipLaunchKernelGGL(k_repredict<1>, dim3(1), dim3(64), 0, s, d_sys, i, which);
    else if (max_nlev <= 4)
        hipLaunchKernelGGL(k_repredict<4>, dim3(1), dim3(64), 0, s, d_sys, i, which);
    else hipLaunchKernelGGL(k_repredict<EDMD_MAX_LEVELS>, dim3(1), dim3(64), 0, s, d_sys, i, which);
    return hipGetLastError();
}

hipError_t edmd_launch_queue_edit(const EdmdSys* d_sys, int max_nlev, int kind, int i, int j,
                                  double t, uint32_t cact, int mode, hipStream_t s) {
    if (max_nlev <= 1)
        hipLaunchKernelGGL(k_queue_edit<1>, dim3(1), dim3(64), 0, s, d_sys, kind, i, j, t, cact, mode);
    else if (max_nlev <= 4)
        hipLaunchKernelGGL(k_queue_edit<4>, dim3(1), dim3(64), 0, s, d_sys, kind, i, j, t, cact, mode);
    else
        hipLaunchKernelGGL(k_queue_edit<EDMD_MAX_LEVELS>, dim3(1), dim3(64), 0, s, d_sys, kind, i, j,
                           t, cact, mode);
    return hipGetLastError();
}

hipError_t edmd_launch_fly_one(const EdmdSys* d_sys, int i, hipStream_t s) {
    hipLaunchKernelGGL(k_fly_one, dim3(1), dim3(1), 0, s, d_sys, i);
    return hipGetLastError();
}

hipError_t edmd_launch_pcf(const double* x, const double* y, const EdmdPart* part, int n, double t,
                           int extrap, double Lx, double Ly, double dr, int nb,
                           unsigned long long* hist, hipStream_t s) {
    const int tiles = (n + 255) / 256;
    hipLaunchKernelGGL(k_pcf, dim3(tiles, tiles), dim3(256), (size_t)nb * sizeof(unsigned int), s,
                       x, y, part, n, t, extrap, Lx, Ly, dr, nb, hist);
    return hipGetLastError();
}

hipError_t edmd_launch_fp64_check(int n, const double* a, const double* b, double* q, double* sq,
                                  hipStream_t s) {
    hipLaunchKernelGGL(k_fp64_check, dim3((n + 255) / 256), dim3(256), 0, s, n, a, b, q, sq);
    return hipGetLastError();
}
