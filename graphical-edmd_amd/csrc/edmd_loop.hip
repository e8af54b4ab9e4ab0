/*
 * Event-loop kernels of libedmd_hip.so for gfx950.
 *
 *   k_run_small, k_run
 *                  persistent event loop: one wavefront per system pops the
 *                  earliest event, applies the reference's handlers
 *                  (EDMD.c:534-610, 2501-2590, 3542-3915, 4657-4713,
 *                  4740-4800, 4828-4923) and re-predicts with all 64 lanes;
 *                  instantiated for the calendar depth and for growing
 *                  systems (the Grow dispatch of EDMD.c:1974-1990)
 *   k_run_lds      the same loop with each system's arrays copied into its
 *                  workgroup's LDS for the duration of the launch
 *
 * Compiled once per variant (EDMD_LOOP_GROW: growing systems, EDMD_LOOP_WALLS:
 * walls, the field or damping), so that the variants build in parallel.
 * Reference line numbers are those of src/EDMD.c.
 */
#define EDMD_DEVICE_ARRAYS 1
#include "edmd_loop.h"
#include "edmd_variants.h"

/* Systems of up to 64^2 disks (calendar depth <= 2): bounded to 128 VGPRs so
 * that four waves share each SIMD and a batch of 4096 replicas is resident
 * at once on 256 CUs. */
template <int ML, bool G, bool W, int WPB = 1>
__global__ __launch_bounds__(64 * WPB, 4) void k_run_small(const EdmdSys* __restrict__ systems,
                                                           EdmdRunArgs ra) {
    /* WPB systems per workgroup, one per wavefront (the launch's systems
     * per workgroup are tuned; the last workgroup may hold fewer) */
    const int sys = WPB > 1 ? (int)blockIdx.x * WPB + wave_in_group() : (int)blockIdx.x;
    if (WPB > 1 && sys >= ra.nsys) return;
    const EdmdSys& S = systems[sys];
    /* G launches run the systems that are growing, the others the rest */
    if ((uni(S.a.st->growing) != 0) != G) return;
    run_loop<ML, G, W, WPB>(S.c, S.a, ra);
}

/* Deeper calendars (large systems, typically one per launch): no register
 * bound, so the path caches stay in registers. */
template <int ML, bool G, bool W>
__global__ __launch_bounds__(64) void k_run(const EdmdSys* __restrict__ systems, EdmdRunArgs ra) {
    const EdmdSys& S = systems[blockIdx.x];
    if ((uni(S.a.st->growing) != 0) != G) return;
    run_loop<ML, G, W>(S.c, S.a, ra);
}

/* ----------------------------------------------------- LDS-resident systems */

#if defined(__HIP_DEVICE_COMPILE__)
#define EDMD_LDS __attribute__((address_space(3)))
#else
#define EDMD_LDS
#endif

/* The arrays of a system whose event loop runs out of LDS.  Everything the
 * loop reads and writes on each event (particles, event slots, calendar
 * nodes, ranks, image counters, cell lists, growth rates) sits in the
 * workgroup's LDS for the whole launch; the per-system record and the
 * output buffers (trace, thermo rows, tape, derivative state) stay in HBM.
 * Fields mean what the fields of EdmdArrays of the same name mean. */
struct EdmdArraysL {
    EdmdPart EDMD_LDS* p;
    EdmdEv EDMD_LDS* e;
    EdmdNode EDMD_LDS* leaf;
    EdmdNode EDMD_LDS* lev[EDMD_MAX_LEVELS];
    int32_t EDMD_LDS* img;
    int32_t EDMD_LDS* ccnt;
    int32_t EDMD_LDS* cslot;
    EdmdState EDMD_GLOBAL* st;
    EdmdTraceRec EDMD_GLOBAL* trace;
    EdmdThermoRow EDMD_GLOBAL* thermo;
    double EDMD_LDS* vr;
    int64_t EDMD_LDS* erank;
    int64_t EDMD_LDS* lrank;
    EdmdTapeRec EDMD_GLOBAL* tape;
    double EDMD_GLOBAL* dv;
    double EDMD_GLOBAL* dtl;
    double EDMD_GLOBAL* otl;
    EdmdDeriv EDMD_GLOBAL* dr;
    int32_t EDMD_GLOBAL* ptype;
    uint32_t EDMD_GLOBAL* mt;
};

/* Copies one array between HBM and LDS with the whole wavefront, in 16-,
 * 8- or 4-byte words as the HBM address and the length allow (LDS offsets
 * are 16-byte aligned; every length is a multiple of 4). */
template <bool IN>
__device__ __forceinline__ void lds_xfer(unsigned char EDMD_LDS* l, const void EDMD_GLOBAL* gv,
                                         uint32_t bytes, int lane) {
    unsigned char EDMD_GLOBAL* g = (unsigned char EDMD_GLOBAL*)gv;
    const uint32_t al = uni((int)((uint32_t)(uintptr_t)g | bytes));
    if ((al & 15) == 0) {
        int4 EDMD_LDS* L = (int4 EDMD_LDS*)l;
        int4 EDMD_GLOBAL* H = (int4 EDMD_GLOBAL*)g;
        for (uint32_t i = lane; i < bytes / 16; i += 64) {
            if (IN) L[i] = H[i]; else H[i] = L[i];
        }
    } else if ((al & 7) == 0) {
        int2 EDMD_LDS* L = (int2 EDMD_LDS*)l;
        int2 EDMD_GLOBAL* H = (int2 EDMD_GLOBAL*)g;
        for (uint32_t i = lane; i < bytes / 8; i += 64) {
            if (IN) L[i] = H[i]; else H[i] = L[i];
        }
    } else {
        int EDMD_LDS* L = (int EDMD_LDS*)l;
        int EDMD_GLOBAL* H = (int EDMD_GLOBAL*)g;
        for (uint32_t i = lane; i < bytes / 4; i += 64) {
            if (IN) L[i] = H[i]; else H[i] = L[i];
        }
    }
}

/* Moves a system's loop arrays into LDS (IN) or back to HBM (!IN); the
 * growth rates are read-only and only come in. */
template <bool IN, bool G>
__device__ __forceinline__ void lds_system(const EdmdConst& C, const EdmdArrays& H,
                                           const EdmdArraysL& A, int lane) {
    const uint32_t n = (uint32_t)C.n, ncell = (uint32_t)(C.ncx * C.ncy);
    lds_xfer<IN>((unsigned char EDMD_LDS*)A.p, H.p, n * 64, lane);
    lds_xfer<IN>((unsigned char EDMD_LDS*)A.e, H.e, n * 32, lane);
    lds_xfer<IN>((unsigned char EDMD_LDS*)A.leaf, H.leaf, n * 16, lane);
    for (int l = 0; l < C.nlev; l++)
        lds_xfer<IN>((unsigned char EDMD_LDS*)A.lev[l], H.lev[l], (uint32_t)C.lsize[l + 1] * 16, lane);
    lds_xfer<IN>((unsigned char EDMD_LDS*)A.erank, H.erank, n * 16, lane);
    lds_xfer<IN>((unsigned char EDMD_LDS*)A.lrank, H.lrank, n * 8, lane);
    lds_xfer<IN>((unsigned char EDMD_LDS*)A.img, H.img, n * 8, lane);
    lds_xfer<IN>((unsigned char EDMD_LDS*)A.ccnt, H.ccnt, ncell * 4, lane);
    lds_xfer<IN>((unsigned char EDMD_LDS*)A.cslot, H.cslot, ncell * (uint32_t)C.cap * 4, lane);
    if (IN && G) lds_xfer<true>((unsigned char EDMD_LDS*)A.vr, H.vr, n * 8, lane);
}

/* One workgroup (one wavefront) per system with the system's loop arrays
 * resident in LDS: they come in from HBM when the launch starts, the event
 * loop runs on them, and they go back when it stops.  The dynamic LDS of
 * the launch holds the largest system's arrays (edmd_lds_layout). */
template <int ML, bool G, bool W>
__global__ __launch_bounds__(64) void k_run_lds(const EdmdSys* __restrict__ systems,
                                                EdmdRunArgs ra) {
    extern __shared__ __align__(64) unsigned char lds_pool[];
    const EdmdSys& S = systems[blockIdx.x];
    const EdmdConst& C = S.c;
    const EdmdArrays& H = S.a;
    const int lane = threadIdx.x;
    if ((uni(H.st->growing) != 0) != G) return;
    const EdmdLdsLayout L = edmd_lds_layout(&C, G ? 1 : 0);
    unsigned char EDMD_LDS* base = (unsigned char EDMD_LDS*)lds_pool;
    /* the pointer table itself lives in LDS: the loop indexes lev[] with
     * run-time levels, which would put a register copy in scratch */
    __shared__ EdmdArraysL A;
    A.p = (EdmdPart EDMD_LDS*)(base + L.p);
    A.e = (EdmdEv EDMD_LDS*)(base + L.e);
    A.leaf = (EdmdNode EDMD_LDS*)(base + L.leaf);
    for (int l = 0; l < EDMD_MAX_LEVELS; l++) A.lev[l] = (EdmdNode EDMD_LDS*)(base + L.lev[l]);
    A.img = (int32_t EDMD_LDS*)(base + L.img);
    A.ccnt = (int32_t EDMD_LDS*)(base + L.ccnt);
    A.cslot = (int32_t EDMD_LDS*)(base + L.cslot);
    A.vr = (double EDMD_LDS*)(base + L.vr);
    A.erank = (int64_t EDMD_LDS*)(base + L.erank);
    A.lrank = (int64_t EDMD_LDS*)(base + L.lrank);
    A.st = H.st;
    A.trace = H.trace;
    A.thermo = H.thermo;
    A.tape = H.tape;
    A.dv = H.dv;
    A.dtl = H.dtl;
    A.otl = H.otl;
    A.dr = H.dr;
    A.ptype = H.ptype;
    A.mt = H.mt;
    WAVE_SYNC();
    lds_system<true, G>(C, H, A, lane);
    WAVE_SYNC();
    run_loop<ML, G, W>(C, A, ra);
    WAVE_SYNC();
    lds_system<false, G>(C, H, A, lane);
}

/* ------------------------------------------------------------ launchers */

template <bool G, bool W>
void EdmdLoopVariant<G, W>::run(const EdmdSys* d_sys, int nsys, int max_nlev, EdmdRunArgs ra,
                                hipStream_t s) {
    ra.nsys = nsys;
    /* the _small loop is bounded to 128 vector registers so that four
     * wavefronts share each SIMD; a batch of at most one system per SIMD
     * gains nothing from that and runs the unbounded loop (the depth-2
     * loop spills to scratch under the bound) */
    const bool few = nsys <= 1024;
    if (max_nlev <= 1 && few) hipLaunchKernelGGL((k_run<1, G, W>), dim3(nsys), dim3(64), 0, s, d_sys, ra);
    else if (max_nlev <= 1) hipLaunchKernelGGL((k_run_small<1, G, W>), dim3(nsys), dim3(64), 0, s, d_sys, ra);
    else if (max_nlev == 2 && few) hipLaunchKernelGGL((k_run<2, G, W>), dim3(nsys), dim3(64), 0, s, d_sys, ra);
    else if (max_nlev == 2) hipLaunchKernelGGL((k_run_small<2, G, W>), dim3(nsys), dim3(64), 0, s, d_sys, ra);
    else if (max_nlev == 3) hipLaunchKernelGGL((k_run<3, G, W>), dim3(nsys), dim3(64), 0, s, d_sys, ra);
    else if (max_nlev <= 4) hipLaunchKernelGGL((k_run<4, G, W>), dim3(nsys), dim3(64), 0, s, d_sys, ra);
    else hipLaunchKernelGGL((k_run<EDMD_MAX_LEVELS, G, W>), dim3(nsys), dim3(64), 0, s, d_sys, ra);
}

template <int WPB>
static void launch_packed(const EdmdSys* d_sys, int nsys, int max_nlev, EdmdRunArgs ra,
                          hipStream_t s) {
    ra.nsys = nsys;
    const dim3 grid((nsys + WPB - 1) / WPB), block(64 * WPB);
    if (max_nlev <= 1) hipLaunchKernelGGL((k_run_small<1, false, false, WPB>), grid, block, 0, s, d_sys, ra);
    else hipLaunchKernelGGL((k_run_small<2, false, false, WPB>), grid, block, 0, s, d_sys, ra);
}

template <bool G, bool W>
void EdmdLoopVariant<G, W>::run_packed(const EdmdSys* d_sys, int nsys, int max_nlev, int wpb,
                                       EdmdRunArgs ra, hipStream_t s) {
    if constexpr (!G && !W) {
        if (wpb == 2) launch_packed<2>(d_sys, nsys, max_nlev, ra, s);
        else launch_packed<4>(d_sys, nsys, max_nlev, ra, s);
    }
}

template <bool G, bool W>
const void* EdmdLoopVariant<G, W>::lds_kernel(int max_nlev) {
    if (max_nlev <= 1) return (const void*)k_run_lds<1, G, W>;
    if (max_nlev == 2) return (const void*)k_run_lds<2, G, W>;
    return nullptr;
}

template <bool G, bool W>
void EdmdLoopVariant<G, W>::run_lds(const EdmdSys* d_sys, int nsys, int max_nlev,
                                    size_t dyn_bytes, EdmdRunArgs ra, hipStream_t s) {
    if (max_nlev <= 1) hipLaunchKernelGGL((k_run_lds<1, G, W>), dim3(nsys), dim3(64), dyn_bytes, s, d_sys, ra);
    else hipLaunchKernelGGL((k_run_lds<2, G, W>), dim3(nsys), dim3(64), dyn_bytes, s, d_sys, ra);
}

template struct EdmdLoopVariant<EDMD_LOOP_GROW, EDMD_LOOP_WALLS>;
