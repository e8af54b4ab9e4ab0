/*
 * Device functions shared by the kernels of libedmd_hip.so for gfx950
 * (CDNA4, 64-lane wavefronts): wave reductions, kinematics, walls,
 * collision and crossing times, the neighbour scans, the calendar and one
 * disk's full prediction.
 *
 * Arithmetic: FP64 throughout, compiled with -ffp-contract=off so that every
 * product and sum is rounded where the reference's C rounds it; division and
 * square root use the compiler's correctly rounded FP64 expansions.
 * Reference line numbers are those of src/EDMD.c.
 */
#ifndef EDMD_DEVICE_H
#define EDMD_DEVICE_H

#ifndef EDMD_DEVICE_ARRAYS
#error "define EDMD_DEVICE_ARRAYS before including edmd_types.h"
#endif
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "edmd_internal.h"
#include "edmd_lanes.h"
#include "edmd_math.h"
#include "edmd_types.h"

#define INF_D __builtin_huge_val()

/* Compiler barrier for memory shared between lanes of one wavefront.  The
 * lanes of a wavefront need no hardware action to see each other's global
 * or LDS stores in program order; this only keeps the compiler from moving
 * memory operations across the point. */
#define WAVE_SYNC() __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront")

/* Marks a value that is equal on every lane.  It stays in vector
 * registers: the event loop has few scalar registers to spare, and pinning
 * these values to them (readfirstlane) made the compiler spill about 130
 * scalar registers into vector-register lanes, whose reloads cost more
 * vector instructions than they saved (8 % of the batched loop's rate). */
__device__ __forceinline__ int uni(int v) { return v; }
__device__ __forceinline__ double uni(double v) { return v; }

/* The wavefront's index within its workgroup, in a scalar register: the
 * system a wavefront runs is addressed through it, so its record is read
 * with scalar loads. */
__device__ __forceinline__ int wave_in_group() {
    return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

__device__ __forceinline__ int64_t uni64(int64_t v) {
    return (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 |
                     (uint32_t)__builtin_amdgcn_readfirstlane((int)v));
}

__device__ __forceinline__ double lane_value(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ int64_t lane_value64(int64_t v, int l) {
    return (int64_t)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(v >> 32), l) << 32 |
                     (uint32_t)__builtin_amdgcn_readlane((int)v, l));
}

/* A word or a double (both words) moved across lanes by a DPP pattern in which
 * every lane has a source: no value to keep, so no move to set one up. */
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
    return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}

template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = dpp_i32<CTRL>((int)b), hi = dpp_i32<CTRL>((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

/* Minimum over the 64 lanes, returned on every lane.  Within each row of
 * 16 lanes: quad swaps (lane ^ 1, lane ^ 2), then the half-row mirror
 * (lane l <-> 7 - l within 8) and the row mirror (l <-> 15 - l), each
 * leaving the minimum of the lanes combined so far on every lane; the four
 * row minima are then read into scalar registers.  No LDS traffic, unlike
 * a shuffle butterfly.  The operands must not be NaN. */
__device__ __forceinline__ double dmin(double a, double b) { return b < a ? b : a; }

__device__ __forceinline__ double wave_min(double v) {
    v = dmin(v, dpp_f64<0xb1>(v));  /* quad_perm [1,0,3,2] */
    v = dmin(v, dpp_f64<0x4e>(v));  /* quad_perm [2,3,0,1] */
    v = dmin(v, dpp_f64<0x141>(v)); /* row_half_mirror */
    v = dmin(v, dpp_f64<0x140>(v)); /* row_mirror */
    const double r0 = lane_value(v, 0), r1 = lane_value(v, 16);
    const double r2 = lane_value(v, 32), r3 = lane_value(v, 48);
    return dmin(dmin(r0, r1), dmin(r2, r3));
}

__device__ __forceinline__ int imin(int a, int b) { return b < a ? b : a; }

/* Minimum of an int over the wave, on every lane: the same DPP pattern as
 * wave_min, each step a single v_min_i32 with a DPP source. */
__device__ __forceinline__ int wave_min_i32(int v) {
    v = imin(v, dpp_i32<0xb1>(v));
    v = imin(v, dpp_i32<0x4e>(v));
    v = imin(v, dpp_i32<0x141>(v));
    v = imin(v, dpp_i32<0x140>(v));
    const int r0 = __builtin_amdgcn_readlane(v, 0), r1 = __builtin_amdgcn_readlane(v, 16);
    const int r2 = __builtin_amdgcn_readlane(v, 32), r3 = __builtin_amdgcn_readlane(v, 48);
    return imin(imin(r0, r1), imin(r2, r3));
}

/* 32-bit key of v - base that never decreases when v increases: the float
 * nearest to v - base (both roundings are monotone), its sign-magnitude
 * bits turned into a signed order (-0 and +0 alike).  v is never NaN. */
__device__ __forceinline__ int order_key(double v, double base) {
    const int b = __float_as_int((float)(v - base));
    const int m = b & 0x7fffffff;
    return b < 0 ? -m : m;
}

/* Two independent int minima over the wave at once: the same DPP steps as
 * wave_min_i32 with the two chains interleaved, so each DPP step's latency
 * is covered by the other chain's step. */
__device__ __forceinline__ void wave_min_i32x2(int& a, int& b) {
    a = imin(a, dpp_i32<0xb1>(a));
    b = imin(b, dpp_i32<0xb1>(b));
    a = imin(a, dpp_i32<0x4e>(a));
    b = imin(b, dpp_i32<0x4e>(b));
    a = imin(a, dpp_i32<0x141>(a));
    b = imin(b, dpp_i32<0x141>(b));
    a = imin(a, dpp_i32<0x140>(a));
    b = imin(b, dpp_i32<0x140>(b));
    const int a0 = __builtin_amdgcn_readlane(a, 0), a1 = __builtin_amdgcn_readlane(a, 16);
    const int a2 = __builtin_amdgcn_readlane(a, 32), a3 = __builtin_amdgcn_readlane(a, 48);
    const int b0 = __builtin_amdgcn_readlane(b, 0), b1 = __builtin_amdgcn_readlane(b, 16);
    const int b2 = __builtin_amdgcn_readlane(b, 32), b3 = __builtin_amdgcn_readlane(b, 48);
    a = imin(imin(a0, a1), imin(a2, a3));
    b = imin(imin(b0, b1), imin(b2, b3));
}

/* ------------------------------------------------------------ kinematics */

/* PBC, EDMD.c:5896-5913 */
__device__ __forceinline__ void min_image(const EdmdConst& C, double& dx, double& dy) {
    /* mihx / mihy are halfLx / halfLy, or +inf across walls (no image) */
    if (dx >= C.mihx) dx -= C.Lx;
    else if (dx < -C.mihx) dx += C.Lx;
    if (dy >= C.mihy) dy -= C.Ly;
    else if (dy < -C.mihy) dy += C.Ly;
}

/* edmd_exp (e^x, the library's own) is in edmd_math.h.  The event loops call
 * the functions below, which only damping and the circular wall need: inlined
 * at each of their places, their constants alone filled the scalar registers,
 * and the loops for walls spilled 300 of them, run or not: 2048 systems of 500
 * disks between walls under the field took 11.2 us a collision with them
 * inlined, 10.5 with calls. */
__device__ __noinline__ double edmd_exp_call(double x) { return edmd_exp(x); }

/* log x from log m = 2 atanh s = 2(s + s^3/3 + ... + s^23/23),
 * s = (m - 1)/(m + 1), x = m 2^e with m in [sqrt(1/2), sqrt(2)), plus
 * e ln2 in two parts; within 4 ulp, the oracle's steps. */
__device__ __noinline__ double edmd_log(double x) {
    if (x != x || x < 0) return __builtin_nan("");
    if (x == 0) return -__builtin_huge_val();
    if (x == __builtin_huge_val()) return x;
    int e;
    double m = frexp(x, &e);
    if (m < 0.70710678118654752) {
        m *= 2;
        e -= 1;
    }
    const double s = (m - 1) / (m + 1), s2 = s * s;
    double q = 1.0 / 23;
#pragma unroll
    for (int n = 21; n >= 1; n -= 2) q = (1.0 / n) + s2 * q;
    const double lm = 2 * s * q;
    return e * 0x1.62e42fefa3800p-1 + (e * 0x1.ef35793c76730p-45 + lm);
}

/* sin and cos of an angle in [-pi, pi] (atan2's range): theta = k pi/2 + r,
 * |r| <= pi/4, pi/2 in three parts (33, 33 and 53 bits, Cody and Waite) so
 * that k times the first two is exact; sin r and cos r from their Taylor
 * series to r^19/19! and r^20/20! in nested form; the quadrant k mod 4
 * picks and signs them.  The oracle runs the same steps; both are within
 * 2 ulp of the C library. */
__device__ __forceinline__ void edmd_sincos(double th, double& sn, double& cs) {
    const double k = rint(th * 0x1.45f306dc9c883p-1); /* th * 2/pi, to nearest */
    const double r = ((th - k * 0x1.921fb54400000p+0) - k * 0x1.0b4611a600000p-34) -
                     k * 0x1.3198a2e037073p-69;
    const double r2 = r * r;
    double ps = 1.0, pc = 1.0;
#pragma unroll
    for (int n = 19; n >= 3; n -= 2) ps = 1.0 - (r2 * ((1.0 / n) * (1.0 / (n - 1)))) * ps;
#pragma unroll
    for (int n = 20; n >= 2; n -= 2) pc = 1.0 - (r2 * ((1.0 / n) * (1.0 / (n - 1)))) * pc;
    const double sr = r * ps, cr = pc;
    switch (((int)k) & 3) {
        case 0: sn = sr; cs = cr; break;
        case 1: sn = cr; cs = -sr; break;
        case 2: sn = -sr; cs = -cr; break;
        default: sn = -cr; cs = sr; break;
    }
}

/* atan z for z in [0, 1]: about 0.4 or 0.8 (atan z = atan c + atan w,
 * w = (z - c)/(1 + z c), |w| <= 0.2), then w (1 - w^2 (1/3 - w^2 (1/5 -
 * ... w^2/23))). */
__device__ __forceinline__ double edmd_atan01(double z) {
    double base = 0, w = z;
    if (z > 0.6) {
        w = (z - 0.8) / (1 + z * 0.8);
        base = 0x1.5977a5103ea93p-1; /* atan(0.8) */
    } else if (z > 0.2) {
        w = (z - 0.4) / (1 + z * 0.4);
        base = 0x1.85a376b677dc0p-2; /* atan(0.4) */
    }
    const double w2 = w * w;
    double q = 1.0 / 23;
#pragma unroll
    for (int n = 21; n >= 3; n -= 2) q = (1.0 / n) - w2 * q;
    return base + w * (1 - w2 * q);
}

/* atan2(y, x) in [-pi, pi], pi/2 and pi as head + tail. */
__device__ __forceinline__ double edmd_atan2(double y, double x) {
    const double ax = fabs(x), ay = fabs(y);
    double a;
    if (ay > ax) a = (0x1.921fb54442d18p+0 - edmd_atan01(ax / ay)) + 0x1.1a62633145c07p-54;
    else if (ax > 0) a = edmd_atan01(ay / ax);
    else a = 0;
    if (__builtin_signbit(x)) a = (0x1.921fb54442d18p+1 - a) + 0x1.1a62633145c07p-53;
    return __builtin_signbit(y) ? -a : a;
}

/* The unit vector (x: cos, y: sin) along (x, y), by its angle. */
__device__ __noinline__ double2 circle_normal(double y, double x) {
    double2 n;
    edmd_sincos(edmd_atan2(y, x), n.y, n.x);
    return n;
}

/* The quartic of the circular wall under the field (quartic.c:27-158):
 * Ferrari's method through the cubic resolvent, step for step as there,
 * with this library's own acos (atan2 of sqrt((1 - t)(1 + t)) and t), cos
 * and cube root (exp(log(x) / 3), the pow with exponent 1./3).  The
 * oracle runs the same steps. */
__device__ __forceinline__ double edmd_cosine(double th) {
    double sn, cs;
    edmd_sincos(th, sn, cs);
    return cs;
}

__device__ __forceinline__ unsigned edmd_solve_p3(double* x, double a, double b, double c) {
    const double a2 = a * a;
    double q = (a2 - 3 * b) / 9;
    const double r = (a * (2 * a2 - 9 * b) + 27 * c) / 54;
    const double r2 = r * r;
    const double q3 = q * q * q;
    if (r2 < q3) {
        double t = r / sqrt(q3);
        if (t < -1) t = -1;
        if (t > 1) t = 1;
        t = edmd_atan2(sqrt((1 - t) * (1 + t)), t);
        a /= 3;
        q = -2 * sqrt(q);
        x[0] = q * edmd_cosine(t / 3) - a;
        x[1] = q * edmd_cosine((t + (2.0 * 3.14159265358979323846)) / 3) - a;
        x[2] = q * edmd_cosine((t - (2.0 * 3.14159265358979323846)) / 3) - a;
        return 3;
    }
    const double m = fabs(r) + sqrt(r2 - q3);
    double A = -(m == 0 ? 0.0 : edmd_exp(edmd_log(m) * (1. / 3)));
    if (r < 0) A = -A;
    const double B = (0 == A ? 0 : q / A);
    a /= 3;
    x[0] = (A + B) - a;
    x[1] = -0.5 * (A + B) - a;
    x[2] = 0.5 * sqrt(3.) * (A - B);
    if (fabs(x[2]) < 1e-12) {
        x[2] = x[1];
        return 2;
    }
    return 1;
}

/* The smallest real root above 1e-9 of a t^4 + b t^3 + c t^2 + d t + e,
 * 1e10 when there is none (smallestRoot, quartic.c:143-157). */
__device__ __noinline__ double edmd_smallest_root(double a, double b, double c, double d,
                                                  double e) {
    const double qa = b / a, qb = c / a, qc = d / a, qd = e / a;
    const double a3 = -qb;
    const double b3 = qa * qc - 4. * qd;
    const double c3 = -qa * qa * qd - qc * qc + 4. * qb * qd;
    double x3[3];
    const unsigned zeroes = edmd_solve_p3(x3, a3, b3, c3);
    double q1, q2, p1, p2, D, sqD, y = x3[0];
    if (zeroes != 1) {
        if (fabs(x3[1]) > fabs(y)) y = x3[1];
        if (fabs(x3[2]) > fabs(y)) y = x3[2];
    }
    D = y * y - 4 * qd;
    if (fabs(D) < 1e-12) {
        q1 = q2 = y * 0.5;
        D = qa * qa - 4 * (qb - y);
        if (fabs(D) < 1e-12) {
            p1 = p2 = qa * 0.5;
        } else {
            sqD = sqrt(D);
            p1 = (qa + sqD) * 0.5;
            p2 = (qa - sqD) * 0.5;
        }
    } else {
        sqD = sqrt(D);
        q1 = (y + sqD) * 0.5;
        q2 = (y - sqD) * 0.5;
        p1 = (qa * q1 - qc) / (q1 - q2);
        p2 = (qc - qa * q2) / (q1 - q2);
    }
    double re[4], im[4];
    D = p1 * p1 - 4 * q1;
    if (D < 0.0) {
        re[0] = -p1 * 0.5;
        im[0] = sqrt(-D) * 0.5;
        re[1] = re[0];
        im[1] = -im[0];
    } else {
        sqD = sqrt(D);
        re[0] = (-p1 + sqD) * 0.5;
        re[1] = (-p1 - sqD) * 0.5;
        im[0] = im[1] = 0.0;
    }
    D = p2 * p2 - 4 * q2;
    if (D < 0.0) {
        re[2] = -p2 * 0.5;
        im[2] = sqrt(-D) * 0.5;
        re[3] = re[2];
        im[3] = -im[2];
    } else {
        sqD = sqrt(D);
        re[2] = (-p2 + sqD) * 0.5;
        re[3] = (-p2 - sqD) * 0.5;
        im[2] = im[3] = 0.0;
    }
    double best = 10000000000;
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (im[i] == 0 && re[i] > 0.000000001 && re[i] < best) best = re[i];
    return best;
}

/* MT19937 (Matsumoto and Nishimura, ACM TOMACS 8(1), 1998), the generator
 * behind the reference's drand (mersenne.c genrand_int32; drand(a, b) =
 * a + (b - a) k / 2^32, EDMD.c:5699-5701): one stream per system, its 624
 * state words and the index of the next one (word 624) in HBM.  Word k of
 * the twist is mt[(k + 397) % 624] ^ (y >> 1) ^ (y odd ? 0x9908b0df : 0)
 * with y the upper bit of mt[k] and the lower 31 of mt[(k + 1) % 624]; in
 * the sequential order of the algorithm the words [0, 227) read only old
 * words, [227, 454) the new [0, 227), [454, 623) the new [227, 396) and
 * word 623 the new words 0 and 396, so each range runs wave-parallel once
 * the one before is stored. */
__device__ __forceinline__ void mt_twist_range(uint32_t EDMD_GLOBAL* mt, int lane, int a, int b) {
    uint32_t nw[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int k = a + lane + 64 * r;
        nw[r] = 0;
        if (k < b) {
            const uint32_t y = (mt[k] & 0x80000000u) | (mt[k + 1 == 624 ? 0 : k + 1] & 0x7fffffffu);
            nw[r] = mt[k + 397 < 624 ? k + 397 : k - 227] ^ (y >> 1) ^ ((y & 1u) ? 0x9908b0dfu : 0u);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int k = a + lane + 64 * r;
        if (k < b) mt[k] = nw[r];
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
}

/* The system's next 32-bit output (uniform). */
template <class AR>
__device__ __forceinline__ uint32_t mt_next(const AR& A, int lane) {
    uint32_t EDMD_GLOBAL* mt = A.mt;
    int idx = uni((int)mt[624]);
    if (idx >= 624) {
        mt_twist_range(mt, lane, 0, 227);
        mt_twist_range(mt, lane, 227, 454);
        mt_twist_range(mt, lane, 454, 623);
        mt_twist_range(mt, lane, 623, 624);
        idx = 0;
    }
    uint32_t y = (uint32_t)uni((int)mt[idx]);
    y ^= (y >> 11);
    y ^= (y << 7) & 0x9d2c5680u;
    y ^= (y << 15) & 0xefc60000u;
    y ^= (y >> 18);
    if (lane == 0) mt[624] = (uint32_t)(idx + 1);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    return y;
}

/* drand(0, hi) of the reference (EDMD.c:5699-5701) on the system's stream. */
template <class AR>
__device__ __forceinline__ double mt_drand0(const AR& A, int lane, double hi) {
    const double g = mt_next(A, lane) * (1.0 / 4294967296.0);
    return (g * (hi - 0.0)) + 0.0;
}

/* sign of EDMD.c:5703-5705: -1, 0 or 1. */
__device__ __forceinline__ double ref_sign(double x) { return (x < 0) ? -1.0 : (double)(x > 0); }

/* logTime, EDMD.c:5709-5721: under damping, the time at which the damped
 * motion has covered what the undamped one covers in t; never when it
 * cannot.  F = false compiles damping out. */
template <bool F>
__device__ __forceinline__ double log_time(const EdmdConst& C, double t) {
    if (!(F && C.damping)) return t;
    const double var = (1 - t * C.gamma);
    if (var < 0) return EDMD_NEVER;
    return -edmd_log(var) / C.gamma;
}

/* The wall part of collisionEventNormal (EDMD.c:2845-2895, no field, mid or
 * circular wall; logTime is the identity without damping): a disk in a
 * boundary cell moving towards the wall gets the time to contact, the
 * starting value of the strict-less minimum over the neighbours.  The x
 * test sets xy = 0 whenever it applies, also when the y wall stays the
 * earlier, as the reference does.  Returns whether a wall time was set. */
__device__ __forceinline__ bool wall_time(const EdmdConst& C, double x, double y, double vx,
                                          double vy, double r, int cx, int cy, double& dt,
                                          int& xy, int typ = 0) {
    bool wall = false;
    dt = EDMD_NEVER;
    xy = 2;
    if ((C.walls & 2) && C.field_on) {
        /* EDMD.c:2846-2860: the bottom wall from the bottom row whatever the
         * velocity; the top wall for any disk moving up (NaN when it cannot
         * reach it) */
        const double f = C.field;
        if (cy == 0) {
            dt = (-vy - sqrt(vy * vy - 2 * f * (y - r))) / f;
            wall = true;
            xy = 1;
        }
        if (vy > 0) {
            const double dt2 = (-vy + sqrt(vy * vy - 2 * f * (y - (C.Ly - r)))) / f;
            if (!__builtin_isnan(dt2) && dt2 < dt) {
                dt = dt2;
                wall = true;
                xy = 1;
            }
        }
    } else if (C.walls & 2) {
        if (cy == 0 && vy < 0) {
            dt = log_time<true>(C, -(y - r) / vy);
            wall = true;
            xy = 1;
        } else if (cy == C.ncy - 1 && vy > 0) {
            dt = log_time<true>(C, (C.Ly - y - r) / vy);
            wall = true;
            xy = 1;
        }
    }
    if (C.walls & 1) {
        if (cx == 0 && vx < 0) {
            const double dw = log_time<true>(C, -(x - r) / vx);
            if (dt > dw) {
                wall = true;
                dt = dw;
            }
            xy = 0;
        } else if (cx == C.ncx - 1 && vx > 0) {
            const double dw = log_time<true>(C, (C.Lx - x - r) / vx);
            if (dt > dw) {
                wall = true;
                dt = dw;
            }
            xy = 0;
        }
    }
    if ((C.walls & 8) && typ == 1) {
        /* the mid wall for the solute (EDMD.c:2897-2915): from within 4 of
         * x = Lx/2, moving towards it */
        const double h = C.Lx / 2;
        if (x > h - 4 && x < h && vx > 0) {
            const double dw = log_time<true>(C, (h - x - r) / vx);
            if (dt > dw) {
                wall = true;
                dt = dw;
            }
            xy = 0;
        } else if (x < h + 4 && x > h && vx < 0) {
            const double dw = log_time<true>(C, ((x - r) - h) / (-vx));
            if (dt > dw) {
                wall = true;
                dt = dw;
            }
            xy = 0;
        }
    }
    if ((C.walls & 4) && C.field_on) {
        /* the circle under the field (EDMD.c:2918-2935): the parabolic
         * flight meets it at the quartic's smallest positive root (y0 about
         * halfLy here) */
        const double y0 = y - C.halfLy, x0 = x - C.halfLx;
        const double e = x0 * x0 + y0 * y0 - (C.halfLx - r) * (C.halfLx - r);
        const double f = C.field;
        const double a = f * f / 4;
        const double b = f * vy;
        const double c = vx * vx + vy * vy + f * y0;
        const double d = 2 * vx * x0 + 2 * vy * y0;
        dt = edmd_smallest_root(a, b, c, d, e);
        wall = true;
        xy = 2;
    } else if (C.walls & 4) {
        /* the circle (EDMD.c:2938-2954, no field): the centre reaches the
         * circle of radius halfLx - r, for every disk; the time replaces
         * the other walls' */
        const double y0 = y - C.halfLx, x0 = x - C.halfLx;
        const double Cc = (x0 * x0 + y0 * y0) - (C.halfLx - r) * (C.halfLx - r);
        const double A = (vx * vx + vy * vy);
        const double B = 2 * (vx * x0 + vy * y0);
        dt = (-B + sqrt(B * B - 4 * A * Cc)) / (2 * A);
        wall = true;
        xy = 2;
    }
    return wall;
}

/* The wall slot of collisionEventGrow (EDMD.c:3118-3153): the surface of a
 * growing disk in a boundary cell closes on the wall at v -/+ vr; no
 * logTime.  dt starts at the growth version's 1e7; as in wall_time, the x
 * test sets xy = 0 whenever it applies. */
__device__ __forceinline__ bool wall_time_grow(const EdmdConst& C, double x, double y, double vx,
                                               double vy, double r, double vr, int cx, int cy,
                                               double& dt, int& xy,
                                               int typ = 0) {
    bool wall = false;
    dt = EDMD_GROW_NONE;
    xy = 2;
    if (C.walls & 2) {
        const double vyp = vy + vr, vym = vy - vr;
        if (cy == 0 && vym < 0) {
            dt = -(y - r) / vym;
            wall = true;
            xy = 1;
        } else if (cy == C.ncy - 1 && vyp > 0) {
            dt = (C.Ly - y - r) / vyp;
            wall = true;
            xy = 1;
        }
    }
    if (C.walls & 1) {
        const double vxp = vx + vr, vxm = vx - vr;
        if (cx == 0 && vxm < 0) {
            const double dw = -(x - r) / vxm;
            if (dt > dw) {
                wall = true;
                dt = dw;
            }
            xy = 0;
        } else if (cx == C.ncx - 1 && vxp > 0) {
            const double dw = (C.Lx - x - r) / vxp;
            if (dt > dw) {
                wall = true;
                dt = dw;
            }
            xy = 0;
        }
    }
    if ((C.walls & 8) && typ == 1) {
        /* EDMD.c:3175-3195 */
        const double h = C.Lx / 2;
        const double vxp = vx + vr, vxm = vx - vr;
        if (x > h - 4 && x < h && vxp > 0) {
            const double dw = (h - x - r) / (vxp);
            if (dt > dw) {
                wall = true;
                dt = dw;
            }
            xy = 0;
        } else if (x < h + 4 && x > h && vxm < 0) {
            const double dw = ((x - r) - h) / (-vxm);
            if (dt > dw) {
                wall = true;
                dt = dw;
            }
            xy = 0;
        }
    }
    if (C.walls & 4) {
        /* EDMD.c:3158-3172: the surface closes on the circle at |v| - vr */
        const double y0 = y - C.halfLx, x0 = x - C.halfLx;
        const double A = vx * vx + vy * vy - vr * vr;
        const double B = 2 * (vx * x0 + vy * y0 + (C.halfLx - r) * vr);
        const double Cc = (x0 * x0 + y0 * y0) - (C.halfLx - r) * (C.halfLx - r);
        dt = (-B + sqrt(B * B - 4 * A * Cc)) / (2 * A);
        wall = true;
        xy = 2;
    }
    return wall;
}

/* PBCinsideCellX/Y, EDMD.c:5922-5936 */
__device__ __forceinline__ double wrap_inside(double d, double half, double L) {
    if (d >= half) return d - L;
    if (d < -half) return d + L;
    return d;
}

/* PBCpostX/Y, EDMD.c:5948-5959 */
__device__ __forceinline__ double wrap_post(double v, double L) {
    if (v < 0) return v + L;
    if (v >= L) return v - L;
    return v;
}

/* PBCcellX/Y, EDMD.c:2110-2124 */
__device__ __forceinline__ int wrap_cell(int a, int nc) {
    if (a < 0) return a + nc;
    if (a >= nc) return a - nc;
    return a;
}

/* freeFlyNormal, EDMD.c:4954-4990, on values held in registers */
__device__ __forceinline__ void fly(const EdmdConst& C, double t, double& x, double& y,
                                    double vx, double vy, double& tl) {
    double dt = t - tl;
    tl = t;
    x += dt * vx;
    y += dt * vy;
    x = wrap_post(x, C.Lx);
    y = wrap_post(y, C.Ly);
}

/* freeFlyNormal for a system with the field (EDMD.c:4957-4963: parabolic
 * in y, vy advanced) or damping (EDMD.c:4965-4975: velocities times
 * exp(-gamma dt)); F = false compiles both out. */
template <bool F>
__device__ __forceinline__ void fly_v(const EdmdConst& C, double t, double& x, double& y,
                                      double& vx, double& vy, double& tl) {
    /* the field first: with both on the flight is the field's alone
     * (EDMD.c:4957-4975), while logTime still applies the damping */
    if (F && C.field_on) {
        const double dt = t - tl;
        tl = t;
        x += dt * vx;
        y += dt * vy + 0.5 * C.field * dt * dt;
        vy += dt * C.field;
        x = wrap_post(x, C.Lx);
        y = wrap_post(y, C.Ly);
    } else if (F && C.damping) {
        const double dt = t - tl;
        tl = t;
        const double g = C.gamma;
        const double ex = edmd_exp_call(-g * dt);
        x += vx / g * (1 - ex);
        y += vy / g * (1 - ex);
        vx *= ex;
        vy *= ex;
        x = wrap_post(x, C.Lx);
        y = wrap_post(y, C.Ly);
    } else {
        fly(C, t, x, y, vx, vy, tl);
    }
}

/* freeFlyGrow, EDMD.c:4992-5007: the radius grows with the flight. */
__device__ __forceinline__ void fly_grow(const EdmdConst& C, double t, double& x, double& y,
                                         double vx, double vy, double& tl, double& rad,
                                         double vr) {
    double dt = t - tl;
    tl = t;
    x += dt * vx;
    y += dt * vy;
    rad += dt * vr;
    x = wrap_post(x, C.Lx);
    y = wrap_post(y, C.Ly);
}

/* collisionTimeNormal, EDMD.c:2661-2723: relative time until contact of the
 * synchronised owner (x1..) with candidate 2 last updated at tl2. */
/* The same with candidate 2's position already flown to t:
 * xt2 = x2 + (t - tl2) * vx2, yt2 likewise (EDMD.c:2667-2671). */
template <bool WRAP = true>
__device__ __forceinline__ double coll_time_at(const EdmdConst& C, double x1, double y1,
                                               double vx1, double vy1, double r1, double xt2,
                                               double yt2, double vx2, double vy2, double r2,
                                               bool& overlap) {
    double dvx = vx2 - vx1;
    double dvy = vy2 - vy1;
    double dx = xt2 - x1;
    double dy = yt2 - y1;
    if (WRAP) min_image(C, dx, dy);
    double b = dx * dvx + dy * dvy;
    if (b > 0) return EDMD_NEVER;
    double v2 = dvx * dvx + dvy * dvy;
    double d = dx * dx + dy * dy - 4 * r1 * r2; /* DIST2, EDMD.c:35-43 */
    double det = b * b - v2 * d;
    if (d < -0.01) overlap = true; /* EDMD.c:2708-2717 */
    if (det < 0) return EDMD_NEVER;
    return (-b - sqrt(det)) / v2;
}

/* collisionTimeNormal as coll_time computes it, without branches: every
 * term is evaluated and the result selected, so a wavefront whose lanes hold
 * different candidates runs one instruction stream.  Bitwise the same
 * result; the overlap test applies where the reference reaches it (b <= 0). */
__device__ __forceinline__ double coll_time_nb(const EdmdConst& C, double t, double x1, double y1,
                                               double vx1, double vy1, double r1, double x2,
                                               double y2, double vx2, double vy2, double tl2,
                                               double r2, bool& overlap) {
    const double lat2 = t - tl2;
    const double dvx = vx2 - vx1;
    const double dvy = vy2 - vy1;
    double dx = (x2 + lat2 * vx2) - x1;
    double dy = (y2 + lat2 * vy2) - y1;
    min_image(C, dx, dy);
    const double b = dx * dvx + dy * dvy;
    const double v2 = dvx * dvx + dvy * dvy;
    const double d = dx * dx + dy * dy - 4 * r1 * r2; /* DIST2, EDMD.c:35-43 */
    const double det = b * b - v2 * d;
    const bool approach = !(b > 0);
    overlap = overlap || (approach && d < -0.01); /* EDMD.c:2708-2717 */
    const double root = (-b - sqrt(det)) / v2;
    return (approach && !(det < 0)) ? root : EDMD_NEVER;
}

__device__ __forceinline__ double coll_time(const EdmdConst& C, double t, double x1, double y1,
                                            double vx1, double vy1, double r1, double x2,
                                            double y2, double vx2, double vy2, double tl2,
                                            double r2, bool& overlap) {
    double lat2 = t - tl2;
    return coll_time_at(C, x1, y1, vx1, vy1, r1, x2 + lat2 * vx2, y2 + lat2 * vy2, vx2, vy2, r2,
                        overlap);
}

/* collisionTimeGrow, EDMD.c:2598-2659 (2D): contact distance
 * DIST(r1, r2(t)) widening at vr1 + vr2; the earlier positive root, or the
 * later one under the reference's 1e-9 rule; an overlap is flagged only
 * when neither root is taken. */
__device__ __forceinline__ double coll_time_grow(const EdmdConst& C, double t, double x1,
                                                 double y1, double vx1, double vy1, double r1,
                                                 double vr1, double x2, double y2, double vx2,
                                                 double vy2, double tl2, double r2, double vr2,
                                                 bool& overlap) {
    double lat2 = t - tl2;
    double dvx = vx2 - vx1;
    double dvy = vy2 - vy1;
    double dvr = vr1 + vr2;
    double dx = (x2 + lat2 * vx2) - x1;
    double dy = (y2 + lat2 * vy2) - y1;
    double dr = sqrt(4 * r1 * (r2 + lat2 * vr2));
    min_image(C, dx, dy);
    double b = dx * dvx + dy * dvy - dvr * dr;
    double v2 = dvx * dvx + dvy * dvy;
    double dist2 = dx * dx + dy * dy;
    double det = b * b - (v2 - dvr * dvr) * (dist2 - dr * dr);
    if (det < 0) return EDMD_NEVER;
    double plus = (-b + sqrt(det)) / (v2 - dvr * dvr);
    double minus = (-b - sqrt(det)) / (v2 - dvr * dvr);
    if (((minus > 0) && (plus > 0) && (minus < plus)) || ((minus > 0) && (plus < 0)))
        return minus;
    else if (((minus > 0) && (plus > 0.000000001) && (plus < minus)) ||
             ((minus < 0) && (plus > 0.000000001)))
        return plus;
    if (dist2 - dr * dr < -0.01) overlap = true; /* EDMD.c:2653-2656 */
    return EDMD_NEVER;
}

/* crossingEventNormal, EDMD.c:2405-2482: absolute crossing time and
 * direction code (1 -x, 2 +x, 3 -y, 4 +y); ties go to y. */
template <bool F = true>
__device__ __forceinline__ void cross_time(const EdmdConst& C, double t, double x, double y,
                                           double vx, double vy, int cx, int cy, double& tout,
                                           int& dir) {
    double tx, ty;
    int xx, yy;
    if (vx < 0) {
        tx = log_time<F>(C, wrap_inside(cx * C.csx - x, C.halfLx, C.Lx) / vx);
        xx = 1;
    } else {
        tx = log_time<F>(C, wrap_inside((1 + cx) * C.csx - x, C.halfLx, C.Lx) / vx);
        xx = 2;
    }
    if (F && C.field_on) {
        /* EDMD.c:2428-2442: up through the top edge when fast enough, else
         * down through the bottom edge */
        const double f = C.field;
        double dy = wrap_inside(y - (1 + cy) * C.csy, C.halfLy, C.Ly);
        if (dy < 0 && vy > sqrt(2 * f * dy)) {
            ty = (-vy + sqrt(vy * vy - 2 * f * dy)) / f;
            yy = 4;
        } else {
            dy = wrap_inside(y - cy * C.csy, C.halfLy, C.Ly);
            ty = (-vy - sqrt(vy * vy - 2 * f * dy)) / f;
            yy = 3;
        }
    } else if (vy < 0) {
        ty = log_time<F>(C, wrap_inside(cy * C.csy - y, C.halfLy, C.Ly) / vy);
        yy = 3;
    } else {
        ty = log_time<F>(C, wrap_inside((1 + cy) * C.csy - y, C.halfLy, C.Ly) / vy);
        yy = 4;
    }
    if (tx < ty) {
        tout = t + tx;
        dir = xx;
    } else {
        tout = t + ty;
        dir = yy;
    }
}

/* Rank of an event scheduled at t_ev with the queue at paulTime = paul after
 * ctr earlier insertions (addEventToQueue, EDMD.c:2144-2170): straight into
 * the tree when t_ev - paulTime < dtPaul, into the overflow list when it is
 * dtPaul * nlists or more ahead, otherwise into a LIFO bucket. */
__device__ __forceinline__ int64_t rank_of(double t_ev, double paul, double dtp, double horizon,
                                           int64_t ctr) {
    const double dt = t_ev - paul;
    /* bucket D - 1 - ctr = D + ~ctr, tree D + ctr, overflow list D + 2^61 +
     * ctr: the low word of D is 0, so the words do not carry (the loop files
     * 4-6 events per collision: no branches, and half the instructions of
     * 64-bit sums) */
    const bool up = (dt < dtp) | (dt >= horizon);
    const uint32_t flip = up ? 0u : 0xffffffffu;
    const uint32_t top = (uint32_t)(EDMD_RANK_DIRECT >> 32) + (dt >= horizon ? 0x20000000u : 0u);
    const uint32_t lo = (uint32_t)ctr ^ flip, hi = ((uint32_t)(ctr >> 32) ^ flip) + top;
    return (int64_t)((uint64_t)hi << 32 | lo);
}

/* Calendar leaf of a particle: its earlier slot by (time, rank) (a NaN key
 * is parked at +inf so that it is never popped), that slot's rank and its
 * event code: the partner for a collision, minus the direction for a
 * crossing. */
struct Leaf {
    double key;
    int64_t rank;
    int aux;
};

__device__ __forceinline__ Leaf make_leaf(double tcoll, int64_t rcoll, double tcross,
                                          int64_t rcross, int partner, int dir) {
    /* non-short-circuit: the compiler keeps a select, not a branch */
    const bool coll = (tcoll < tcross) | ((tcoll == tcross) & (rcoll < rcross));
    Leaf L;
    const double k = coll ? tcoll : tcross;
    L.key = (k == k) ? k : INF_D;
    L.rank = coll ? rcoll : rcross;
    L.aux = coll ? partner : -dir;
    return L;
}

__device__ __forceinline__ bool before(double ka, int64_t ra, double kb, int64_t rb) {
    return (ka < kb) | ((ka == kb) & (ra < rb));
}

/* ------------------------------------------------------------ predictions */

/* Sequential neighbour scan for one particle (one lane): strict-less minimum
 * in the reference's order, y offset outer, x offset inner, newest list
 * entry first (EDMD.c:2959-3003).  Returns the relative time; NEVER and
 * partner 0 when no candidate qualifies (EDMD.c:2830-2831). */
template <bool G, bool W = true, class AR>
__device__ __forceinline__ double predict_seq(const EdmdConst& C, const AR& A, double t,
                                              int p, const EdmdPart& o, int& partner,
                                              bool& overlap) {
    /* collisionEventGrow (EDMD.c:3104-3230, no walls) starts from 1e7 */
    double dt = G ? EDMD_GROW_NONE : EDMD_NEVER;
    int best = 0;
    const double ovr = G ? A.vr[p] : 0.0;
    int xy = 2;
    bool wall = false;
    const int typ = (W && (C.walls & 8)) ? A.ptype[p] : 0;
    if (W && !G && C.walls)
        wall = wall_time(C, o.x, o.y, o.vx, o.vy, o.rad, o.cx, o.cy, dt, xy, typ);
    if (W && G && C.walls)
        wall = wall_time_grow(C, o.x, o.y, o.vx, o.vy, o.rad, ovr, o.cx, o.cy, dt, xy, typ);
    for (int j = -1; j <= 1; ++j) {
        int row = wrap_cell(o.cy + j, C.ncy) * C.ncx;
        for (int k = -1; k <= 1; ++k) {
            int c = row + wrap_cell(o.cx + k, C.ncx);
            int cnt = A.ccnt[c];
            const auto sl = A.cslot + (size_t)c * C.cap;
            for (int s = cnt - 1; s >= 0; --s) {
                int q = sl[s];
                if (q == p) continue;
                EdmdPart c2 = A.p[q];
                if (W && !G && (C.field_on || C.damping)) {
                    /* collisionTimeNormal flies the neighbour first under
                     * the field or damping, a state update (EDMD.c:2664-2666) */
                    fly_v<true>(C, t, c2.x, c2.y, c2.vx, c2.vy, c2.tl);
                    const auto w = A.p + q;
                    w->x = c2.x;
                    w->y = c2.y;
                    w->vx = c2.vx;
                    w->vy = c2.vy;
                    w->tl = c2.tl;
                }
                double tt;
                if (G)
                    tt = coll_time_grow(C, t, o.x, o.y, o.vx, o.vy, o.rad, ovr, c2.x, c2.y, c2.vx,
                                        c2.vy, c2.tl, c2.rad, A.vr[q], overlap);
                else
                    tt = log_time<W && !G>(
                        C, coll_time(C, t, o.x, o.y, o.vx, o.vy, o.rad, c2.x, c2.y, c2.vx, c2.vy,
                                     c2.tl, c2.rad, overlap));
                if (dt > tt) {
                    dt = tt;
                    best = q;
                    wall = false;
                }
            }
        }
    }
    partner = wall ? EDMD_WALL_CODE(xy) : best;
    return dt;
}

/* ------------------------------------------------------------ calendar */

/* Minimum over the wave by (key, rank), carrying the leaf and the event
 * code.  A node's rank is that of its leaf (lrank[leaf]); ranks are read
 * only when several lanes hold the minimum key, which is rare.  Keys are
 * never NaN; among +inf keys (padding, parked events) the lowest lane wins.
 * base: a time near the keys (the current time), for the 32-bit search. */
/* The part of wave_argmin after the key search: kk is this lane's order
 * key, mkk the minimum key over the wave. */
template <class AR>
__device__ __forceinline__ void wave_argmin_finish(const AR& A, int kk, int mkk, double& k,
                                                   int& i, int& x) {
    const uint64_t near = __ballot(kk == mkk);
    double mk;
    uint64_t tied;
    if (__popcll(near) == 1) {
        tied = near;
        mk = lane_value(k, (int)__builtin_ctzll(near));
    } else {
        const double kv = (kk == mkk) ? k : INF_D;
        mk = wave_min(kv);
        tied = __ballot(kv == mk);
    }
    int w = (int)__builtin_ctzll(tied);
    if (__popcll(tied) > 1 && mk < INF_D) {
        /* equal keys: the earlier in the reference's queue (lower rank) */
        /* loaded by every lane (padding lanes read leaf 0) and selected,
         * not loaded under a divergent branch */
        const bool tie = lane_in(tied);
        const int64_t rl = A.lrank[tie ? i : 0];
        int64_t r = tie ? rl : INT64_MAX;
        int l = tie ? (int)(threadIdx.x & 63) : 64;
#pragma unroll
        for (int m = 1; m < 64; m <<= 1) {
            const long long orr = __shfl_xor((long long)r, m, 64);
            const int ol = __shfl_xor(l, m, 64);
            if (orr < r || (orr == r && ol < l)) {
                r = orr;
                l = ol;
            }
        }
        w = uni(l);
    }
    k = mk;
    i = __builtin_amdgcn_readlane(i, w);
    x = __builtin_amdgcn_readlane(x, w);
}

template <class AR>
__device__ __forceinline__ void wave_argmin(const AR& A, double base, double& k, int& i,
                                            int& x) {
    const int kk = order_key(k, base);
    wave_argmin_finish(A, kk, wave_min_i32(kk), k, i, x);
}

/* wave_argmin of two independent (key, leaf, code) sets, the key searches
 * interleaved; each result is the one wave_argmin gives for its set. */
template <class AR>
__device__ __forceinline__ void wave_argmin2(const AR& A, double base, double& ka, int& ia,
                                             int& xa, double& kb, int& ib, int& xb) {
    const int kka = order_key(ka, base), kkb = order_key(kb, base);
    int ma = kka, mb = kkb;
    wave_min_i32x2(ma, mb);
    wave_argmin_finish(A, kka, ma, ka, ia, xa);
    wave_argmin_finish(A, kkb, mb, kb, ib, xb);
}

/* Level l of the calendar: the leaves for l = 0, else nodes of level l. */
template <class AR>
__device__ __forceinline__ auto level(const AR& A, int l) -> decltype(A.leaf) {
    return l == 0 ? A.leaf : A.lev[l - 1];
}

/* Earliest pending particle event: minimum of the top level, read from
 * `top` (the LDS copy the event loop keeps, or the level in HBM). */
template <class AR>
__device__ __forceinline__ void top_min(const EdmdConst& C, const AR& A, int lane,
                                        const EdmdNode* top, double base, double& key, int& leaf,
                                        int& aux) {
    double k = INF_D;
    int i = 0x7fffffff, x = 0;
    if (lane < C.lsize[C.nlev]) {
        const EdmdNode nd = top[lane];
        k = nd.key;
        i = nd.idx;
        x = nd.aux;
    }
    wave_argmin(A, base, k, i, x);
    key = k;
    leaf = uni(i);
    aux = uni(x);
}

/* The 64 children of every node on the calendar paths of up to two leaves,
 * read in one round trip before the event changes anything.  ML bounds the
 * number of levels above the leaves. */
template <int ML>
struct PathCache {
    double k[2][ML];
    int i[2][ML];
    int x[2][ML];
};

template <int ML, class AR>
__device__ __forceinline__ void path_prefetch(const EdmdConst& C, const AR& A, int lane,
                                              int pA, int pB, PathCache<ML>& P) {
#pragma unroll
    for (int l = 0; l < ML; ++l) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int p = h ? pB : pA;
            double k = INF_D;
            int i = 0x7fffffff, x = 0;
            if (l < C.nlev && p >= 0) {
                const int c = ((p >> (6 * (l + 1))) << 6) + lane;
                if (c < C.lsize[l]) {
                    const EdmdNode nd = level(A, l)[c];
                    k = nd.key;
                    i = nd.idx;
                    x = nd.aux;
                }
            }
            P.k[h][l] = k;
            P.i[h][l] = i;
            P.x[h][l] = x;
        }
    }
}

/* Stores leaf p with its rank. */
template <class AR>
__device__ __forceinline__ void leaf_store(const AR& A, int lane, int p, const Leaf& L) {
    if (lane == 0) {
        EdmdNode n;
        n.key = L.key;
        n.idx = p;
        n.aux = L.aux;
        A.leaf[p] = n;
        A.lrank[p] = L.rank;
    }
}

/* Recomputes every node on the paths of pA (and pB >= 0), whose new leaves
 * (keys kA, kB, event codes xA, xB) the caller has stored with their ranks,
 * from the prefetched children, substituting the freshly computed path
 * nodes; where the paths meet one node takes both.  With `top` (the event
 * loop's LDS copy of the top level) the top-level nodes are written there
 * instead of to HBM. */
template <int ML, class AR>
__device__ __forceinline__ void path_update(const EdmdConst& C, const AR& A, int lane,
                                            const PathCache<ML>& P, int pA, double kA, int xA,
                                            int pB, double kB, int xB, EdmdNode* top,
                                            double base) {
    if (top && C.nlev == 0 && lane == 0) {
        EdmdNode n;
        n.key = kA;
        n.idx = pA;
        n.aux = xA;
        top[pA] = n;
        if (pB >= 0) {
            n.key = kB;
            n.idx = pB;
            n.aux = xB;
            top[pB] = n;
        }
    }
    WAVE_SYNC();
    int iA = pA, iB = pB;
    int cA = pA, cB = pB;
#pragma unroll
    for (int l = 0; l < ML; ++l) {
        if (l >= C.nlev) break;
        const int gA = cA >> 6;
        const int gB = pB >= 0 ? (cB >> 6) : -1;
        int c = (gA << 6) + lane;
        double k = P.k[0][l];
        int i = P.i[0][l], x = P.x[0][l];
        if (c == cA) { k = kA; i = iA; x = xA; }
        else if (pB >= 0 && c == cB) { k = kB; i = iB; x = xB; }
        double nkA, nkB;
        int niA, nxA, niB, nxB;
        if (pB >= 0 && gB != gA) {
            /* two different nodes: both minima at once */
            const int c2 = (gB << 6) + lane;
            double k2 = P.k[1][l];
            int i2 = P.i[1][l], x2 = P.x[1][l];
            if (c2 == cB) { k2 = kB; i2 = iB; x2 = xB; }
            wave_argmin2(A, base, k, i, x, k2, i2, x2);
            nkB = k2;
            niB = uni(i2);
            nxB = uni(x2);
            nkA = k;
            niA = uni(i);
            nxA = uni(x);
        } else {
            wave_argmin(A, base, k, i, x);
            nkA = k;
            niA = uni(i);
            nxA = uni(x);
            nkB = nkA;
            niB = niA;
            nxB = nxA;
        }
        if (lane == 0) {
            EdmdNode n;
            n.key = nkA;
            n.idx = niA;
            n.aux = nxA;
            EdmdNode nb;
            nb.key = nkB;
            nb.idx = niB;
            nb.aux = nxB;
            const bool two = pB >= 0 && gB != gA;
            if (top && l + 1 == C.nlev) {
                top[gA] = n;
                if (two) top[gB] = nb;
            } else {
                A.lev[l][gA] = n;
                if (two) A.lev[l][gB] = nb;
            }
        }
        kA = nkA; iA = niA; xA = nxA;
        kB = nkB; iB = niB; xB = nxB;
        cA = gA;
        cB = gB;
    }
    WAVE_SYNC();
}

/* Sequential minimum over the children of node g of level l (l >= 1) by
 * (key, rank).  Every node holds a real leaf index (0 <= idx < n), so each
 * child's rank is loaded unconditionally and the winner chosen by selects:
 * a rank load under a divergent branch here has been compiled into code
 * that kept the previous winner's event code on a tie (gfx950, ROCm 7.2). */
template <class AR>
__device__ __forceinline__ void node_min(const EdmdConst& C, const AR& A, int l, int g) {
    int lo = g << 6;
    int hi = lo + 64;
    if (hi > C.lsize[l - 1]) hi = C.lsize[l - 1];
    const auto ch = level(A, l - 1);
    const EdmdNode b0 = ch[lo];
    double bk = b0.key;
    int bi = b0.idx, bx = b0.aux;
    int64_t br = A.lrank[bi];
    for (int c = lo + 1; c < hi; ++c) {
        const EdmdNode nd = ch[c];
        const int64_t r = A.lrank[nd.idx];
        const bool take = nd.key < bk || (nd.key == bk && bk < INF_D && r < br);
        bk = take ? nd.key : bk;
        bi = take ? nd.idx : bi;
        bx = take ? nd.aux : bx;
        br = take ? r : br;
    }
    EdmdNode best;
    best.key = bk;
    best.idx = bi;
    best.aux = bx;
    A.lev[l - 1][g] = best;
}

/* ------------------------------------------------------------ sweep */

/* One particle's full prediction (crossing + collision) written to its two
 * slots and its leaf; the particle is assumed synchronised at t.  G selects
 * the growth functions.  The slots are scheduled as insertions number
 * ctr_cross and ctr_coll with the queue at paulTime = paul.  stop_grow: the
 * partner counter recorded is the one stopGrow's interleaved loop sees
 * (EDMD.c:4770-4776: every counter goes 0 -> 1 in particle order, each disk
 * predicting right after its own increment), i.e. 1 for a partner of lower
 * or equal index, else 0. */
template <bool G, bool W = true, class AR>
__device__ __forceinline__ bool sweep_one(const EdmdConst& C, const AR& A, double t, int p,
                                          double paul, int64_t ctr_cross, int64_t ctr_coll,
                                          bool stop_grow = false) {
    const EdmdPart o = A.p[p];
    double tc;
    int dir;
    /* crossingEventGrow while growing: no field, no logTime */
    cross_time<W && !G>(C, t, o.x, o.y, o.vx, o.vy, o.cx, o.cy, tc, dir);
    bool ov = false;
    int partner;
    double dt = predict_seq<G, W>(C, A, t, p, o, partner, ov);
    double tk = t + dt;
    EdmdEv e;
    e.tcoll = tk;
    e.tcross = tc;
    e.partner = partner;
    e.cact = stop_grow ? (partner <= p ? 1u : 0u) : (partner >= 0 ? A.p[partner].coll : 0u);
    e.dir = dir;
    e.pad = 0;
    A.e[p] = e;
    const int64_t rk = rank_of(tk, paul, C.dtp, C.horizon, ctr_coll);
    const int64_t rx = rank_of(tc, paul, C.dtp, C.horizon, ctr_cross);
    A.erank[2 * p] = rk;
    A.erank[2 * p + 1] = rx;
    const Leaf L = make_leaf(tk, rk, tc, rx, partner, dir);
    EdmdNode n;
    n.key = L.key;
    n.idx = p;
    n.aux = L.aux;
    A.leaf[p] = n;
    A.lrank[p] = L.rank;
    return ov;
}

#endif
