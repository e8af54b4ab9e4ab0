/*
 * A system's loop arrays resident in its workgroup's LDS for one launch.
 */
#ifndef EDMD_LDS_H
#define EDMD_LDS_H

#include "edmd_device.h"

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

/* Copies one array between HBM and LDS with the whole group of NT threads, in
 * 16-, 8- or 4-byte words as the HBM address and the length allow (LDS offsets
 * are 16-byte aligned; every length is a multiple of 4). */
template <bool IN, int NT>
__device__ __forceinline__ void lds_xfer(unsigned char EDMD_LDS* l, const void EDMD_GLOBAL* gv,
                                         uint32_t bytes, int tid) {
    unsigned char EDMD_GLOBAL* g = (unsigned char EDMD_GLOBAL*)gv;
    const uint32_t al = uni((int)((uint32_t)(uintptr_t)g | bytes));
    if ((al & 15) == 0) {
        int4 EDMD_LDS* L = (int4 EDMD_LDS*)l;
        int4 EDMD_GLOBAL* H = (int4 EDMD_GLOBAL*)g;
        for (uint32_t i = tid; i < bytes / 16; i += NT) {
            if (IN) L[i] = H[i]; else H[i] = L[i];
        }
    } else if ((al & 7) == 0) {
        int2 EDMD_LDS* L = (int2 EDMD_LDS*)l;
        int2 EDMD_GLOBAL* H = (int2 EDMD_GLOBAL*)g;
        for (uint32_t i = tid; i < bytes / 8; i += NT) {
            if (IN) L[i] = H[i]; else H[i] = L[i];
        }
    } else {
        int EDMD_LDS* L = (int EDMD_LDS*)l;
        int EDMD_GLOBAL* H = (int EDMD_GLOBAL*)g;
        for (uint32_t i = tid; i < bytes / 4; i += NT) {
            if (IN) L[i] = H[i]; else H[i] = L[i];
        }
    }
}

/* Moves a system's loop arrays into LDS (IN) or back to HBM (!IN); the
 * growth rates are read-only and only come in. */
template <bool IN, bool G, int NT>
__device__ __forceinline__ void lds_system(const EdmdConst& C, const EdmdArrays& H,
                                           const EdmdArraysL& A, int tid) {
    const uint32_t n = (uint32_t)C.n, ncell = (uint32_t)(C.ncx * C.ncy);
    lds_xfer<IN, NT>((unsigned char EDMD_LDS*)A.p, H.p, n * 64, tid);
    lds_xfer<IN, NT>((unsigned char EDMD_LDS*)A.e, H.e, n * 32, tid);
    lds_xfer<IN, NT>((unsigned char EDMD_LDS*)A.leaf, H.leaf, n * 16, tid);
    for (int l = 0; l < C.nlev; l++)
        lds_xfer<IN, NT>((unsigned char EDMD_LDS*)A.lev[l], H.lev[l], (uint32_t)C.lsize[l + 1] * 16, tid);
    lds_xfer<IN, NT>((unsigned char EDMD_LDS*)A.erank, H.erank, n * 16, tid);
    lds_xfer<IN, NT>((unsigned char EDMD_LDS*)A.lrank, H.lrank, n * 8, tid);
    lds_xfer<IN, NT>((unsigned char EDMD_LDS*)A.img, H.img, n * 8, tid);
    lds_xfer<IN, NT>((unsigned char EDMD_LDS*)A.ccnt, H.ccnt, ncell * 4, tid);
    lds_xfer<IN, NT>((unsigned char EDMD_LDS*)A.cslot, H.cslot, ncell * (uint32_t)C.cap * 4, tid);
    if (IN && G) lds_xfer<true, NT>((unsigned char EDMD_LDS*)A.vr, H.vr, n * 8, tid);
}

/* Lays the arrays of a system out in its workgroup's LDS (edmd_lds_layout);
 * the others stay in HBM.  Returns the bytes used. */
template <bool G>
__device__ __forceinline__ uint32_t lds_carve(const EdmdConst& C, const EdmdArrays& H,
                                              unsigned char EDMD_LDS* base, EdmdArraysL& A) {
    const EdmdLdsLayout L = edmd_lds_layout(&C, G ? 1 : 0);
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
    return L.total;
}

#endif
