/* Launchers of the event loop's variants: G, the systems that are growing;
 * W, walls, the field or damping.  Each variant is a translation unit of
 * its own (edmd_loop.hip). */
#ifndef EDMD_VARIANTS_H
#define EDMD_VARIANTS_H

#include "edmd_internal.h"

template <bool G, bool W>
struct EdmdLoopVariant {
    static void run(const EdmdSys* d_sys, int nsys, int max_nlev, EdmdRunArgs ra, hipStream_t s);
    /* Systems of calendar depth <= 2 without growth, walls, field or
     * damping, wpb (2 or 4) systems per workgroup. */
    static void run_packed(const EdmdSys* d_sys, int nsys, int max_nlev, int wpb, EdmdRunArgs ra,
                           hipStream_t s);
    /* The LDS-resident loop exists for calendars of depth <= 2 (up to 4096
     * disks, far more than one workgroup's LDS holds). */
    static const void* lds_kernel(int max_nlev);
    static void run_lds(const EdmdSys* d_sys, int nsys, int max_nlev, size_t dyn_bytes,
                        EdmdRunArgs ra, hipStream_t s);
};

/* The wide loop (edmd_wide.hip): one system per workgroup of 4, 8 or
 * 16 wavefronts; place: EDMD_WIDE_*. */
template <bool G, bool W>
struct EdmdWideVariant {
    static const void* kernel(int waves, int place);
    static hipError_t run(int waves, int place, const EdmdSys* d_sys, int nsys, size_t dyn_bytes,
                          EdmdRunArgs ra, hipStream_t s);
};

#endif
