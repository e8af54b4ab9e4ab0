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
#include "edmd_lds.h"
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
    /* the pointer table itself lives in LDS: the loop indexes lev[] with
     * run-time levels, which would put a register copy in scratch */
    __shared__ EdmdArraysL A;
    lds_carve<G>(C, H, (unsigned char EDMD_LDS*)lds_pool, A);
    WAVE_SYNC();
    lds_system<true, G, 64>(C, H, A, lane);
    WAVE_SYNC();
    run_loop<ML, G, W>(C, A, ra);
    WAVE_SYNC();
    lds_system<false, G, 64>(C, H, A, lane);
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
