/*
 * g(r) (calculate_pcf, pcf.c:16-75) on gfx950: the histogram of minimum-image
 * pair distances below rmax = dr * nb, one count per unordered pair (the
 * reference adds 2.0 per pair; the host doubles the counts).
 *
 *   k_pcf_clear  counts of the result and of the sort set to zero
 *   k_pcf_count  each disk's place in its cell of a grid over the box
 *   k_pcf_place  positions (free-flown to the system time where asked) in the
 *                order of a curve through the grid
 *   k_pcf_boxes  the bounding box of every 64 of them
 *   k_pcf_pairs  the histogram: 64 x 64 tiles of the pair triangle, tiles
 *                whose boxes lie further apart than rmax left out
 *
 * The reference takes all n^2 / 2 pairs, 1.88 ms a call at n = 60000
 * on the card; now 60 us of pairs and 0.24 ms a call, most of it allocation
 * and copies.  Only n pi rho rmax^2 / 2 pairs can count (8.4 million
 * of 1.8 billion at rmax = 10 diameters, phi = 0.7); of the compact tiles' pairs
 * about one in four does.  The order does not matter: a pair's distance is the
 * same bits either way round, and counts are whole numbers.
 */
#define EDMD_DEVICE_ARRAYS 1
#include "edmd_device.h"

#define PCF_GRID 64 /* cells a side of the sorting grid */
#define PCF_SORT_THREADS 1024
#define PCF_WAVES 16

/* Position of disk q: host arrays' copies, or the disk's record, free-flown
 * to t without being stored when extrap is set. */
__device__ __forceinline__ double2 pcf_position(const double* px, const double* py,
                                                const EdmdPart* part, int q, double t, int extrap,
                                                double Lx, double Ly) {
    if (!part) return make_double2(px[q], py[q]);
    const EdmdPart r = part[q];
    double x = r.x, y = r.y;
    if (extrap) {
        const double dt = t - r.tl;
        x += dt * r.vx;
        y += dt * r.vy;
        x = wrap_post(x, Lx);
        y = wrap_post(y, Ly);
    }
    return make_double2(x, y);
}

__device__ __forceinline__ int pcf_side(double v, double f) {
    const double c = v * f;
    return c >= PCF_GRID - 1 ? PCF_GRID - 1 : (c > 0 ? (int)c : 0); /* NaN: 0 */
}

/* The cell's place on Hilbert's curve through the grid: 64 disks in a row lie
 * in a few adjoining cells, where Z order's runs cross the box now and then
 * (k_pcf_pairs at n = 60000: 117 us
 * in Z order, 81 us so). */
__device__ __forceinline__ int pcf_cell(double2 p, double fx, double fy) {
    int x = pcf_side(p.x, fx), y = pcf_side(p.y, fy), c = 0;
#pragma unroll
    for (int half = PCF_GRID / 2; half > 0; half >>= 1) {
        const bool right = x >= half, upper = y >= half;
        c = 4 * c + (upper ? (right ? 2 : 1) : (right ? 3 : 0));
        x -= right ? half : 0;
        y -= upper ? half : 0;
        if (!upper) { /* the curve's lower quarters are transposed, the last one about the other diagonal */
            const int u = right ? half - 1 - y : y;
            y = right ? half - 1 - x : x;
            x = u;
        }
    }
    return c;
}

__global__ __launch_bounds__(256) void k_pcf_clear(unsigned long long* __restrict__ hist, int nb,
                                                  int* __restrict__ cnt, int cells) {
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q < nb) hist[q] = 0;
    if (q < cells) cnt[q] = 0;
}

/* Counting sort.  By one workgroup with its counters in LDS it took 69 us at
 * n = 60000 (LDS atomics of a single CU); over the chip clear,
 * count and place take 17 us together.  The place a disk gets in its cell may differ from run to
 * run; the counts of pairs do not. */
__global__ __launch_bounds__(256) void k_pcf_count(const double* __restrict__ px,
                                                  const double* __restrict__ py,
                                                  const EdmdPart* __restrict__ part, int n, double t,
                                                  int extrap, double Lx, double Ly,
                                                  int* __restrict__ cnt, int* __restrict__ place) {
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q >= n) return;
    const double2 p = pcf_position(px, py, part, q, t, extrap, Lx, Ly);
    place[q] = atomicAdd(&cnt[pcf_cell(p, PCF_GRID / Lx, PCF_GRID / Ly)], 1);
}

/* Every workgroup sums the cells' counts for itself (16 KB of L2). */
__global__ __launch_bounds__(PCF_SORT_THREADS) void k_pcf_place(
    const double* __restrict__ px, const double* __restrict__ py,
    const EdmdPart* __restrict__ part, int n, double t, int extrap, double Lx, double Ly,
    const int* __restrict__ cnt, const int* __restrict__ place, double2* __restrict__ out) {
    constexpr int CELLS = PCF_GRID * PCF_GRID, PER = CELLS / PCF_SORT_THREADS;
    __shared__ int start[CELLS];
    __shared__ int sums[PCF_SORT_THREADS / 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int q = blockIdx.x * PCF_SORT_THREADS + tid;
    int own[PER], sum = 0;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        own[k] = cnt[PER * tid + k];
        sum += own[k];
    }
    int incl = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int u = __shfl_up(incl, d, 64);
        if (lane >= d) incl += u;
    }
    if (lane == 63) sums[tid >> 6] = incl;
    __syncthreads();
    int base = incl - sum;
    for (int w = 0; w < (tid >> 6); ++w) base += sums[w];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        start[PER * tid + k] = base;
        base += own[k];
    }
    __syncthreads();
    if (q >= n) return;
    const double2 p = pcf_position(px, py, part, q, t, extrap, Lx, Ly);
    out[start[pcf_cell(p, PCF_GRID / Lx, PCF_GRID / Ly)] + place[q]] = p;
}

/* Bounding boxes {x min, x max, y min, y max} of every 64 positions (NaN
 * positions, which never count, left out). */
__global__ __launch_bounds__(256) void k_pcf_boxes(const double2* __restrict__ pos, int n,
                                                  double4* __restrict__ box) {
    const int tile = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int q = tile * 64 + lane;
    if (tile * 64 >= n) return;
    const double2 p = pos[q < n ? q : tile * 64];
    double lx = p.x, hx = p.x, ly = p.y, hy = p.y;
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        lx = fmin(lx, __shfl_xor(lx, m, 64));
        hx = fmax(hx, __shfl_xor(hx, m, 64));
        ly = fmin(ly, __shfl_xor(ly, m, 64));
        hy = fmax(hy, __shfl_xor(hy, m, 64));
    }
    if (lane == 0) box[tile] = make_double4(lx, hx, ly, hy);
}

/* Least minimum-image distance along one axis of points in [a0, a1] and
 * [b0, b1]: the image taken is d, d - L or d + L of the difference d, so the
 * distance is at least that of the nearest of 0, L and -L from d's range. */
__device__ __forceinline__ double pcf_apart(double a0, double a1, double b0, double b1, double L) {
    const double lo = b0 - a1, hi = b1 - a0;
    auto from = [&](double v) { return fmax(0.0, fmax(lo - v, v - hi)); };
    return fmin(from(0.0), fmin(from(L), from(-L)));
}

/* The pairs of one staged tile with this lane's disk a (act: there is one);
 * only the tile's disks after `first` (in the tile's own pairs, j > i).  WRAP
 * = false: no difference reaches half the box, so no image is taken.
 *
 * A pair's bin is (int)(sqrt(d2) / dr) with the reference's roundings: the
 * 64-bit square root and division take it only where a 32-bit quotient (error
 * below 3.2e-7 of it: four roundings of half a unit, a root good to one) lies
 * within `tol` = 1e-6 + 4e-7 nb of a whole number, or at the bins' end.  With the
 * 64-bit root and division for every pair the kernel takes 88.5 us for 59.4
 * (60000 disks, 500 bins up to 10 diameters). */
template <bool WRAP>
__device__ __forceinline__ void pcf_tile(const double2* stage, int jn, double2 a, bool act,
                                         int first, double Lx, double Ly, double dr, float inv,
                                         float tol, double rmax, double near2, int nb,
                                         unsigned int* h) {
    const double halfLx = Lx / 2, halfLy = Ly / 2;
    for (int k0 = 0; k0 < jn; k0 += 4) {
        double2 b[4];
        double d2[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) b[u] = stage[k0 + u]; /* 64 places, whatever jn */
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            double dx = b[u].x - a.x;
            double dy = b[u].y - a.y;
            if (WRAP) {
                if (dx >= halfLx) dx -= Lx;
                else if (dx < -halfLx) dx += Lx;
                if (dy >= halfLy) dy -= Ly;
                else if (dy < -halfLy) dy += Ly;
            }
            d2[u] = dx * dx + dy * dy;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int k = k0 + u;
            if (d2[u] <= near2 && act && k > first && k < jn) {
                const float q = __builtin_amdgcn_sqrtf((float)d2[u]) * inv;
                int bin = (int)q;
                if (!(fabsf(q - rintf(q)) > tol && q < nb)) {
                    const double r = sqrt(d2[u]);
                    bin = r < rmax ? (int)(r / dr) : nb;
                }
                if (bin < nb) atomicAdd(&h[bin], 1u);
            }
        }
    }
}

/* One workgroup of 16 wavefronts counts into one LDS histogram over its share
 * of the tiles (its counts are added to the result once, at the end), S slices
 * a tile where there are few.  Of the tiles right of tile I in the triangle
 * each wavefront tests 64 boxes; those kept are dealt to the wavefronts, and a
 * wavefront holds I's disks one a lane and walks the other tile's through its
 * LDS stage. */
template <bool SORTED>
__global__ __launch_bounds__(64 * PCF_WAVES) void k_pcf_pairs(
    const double2* __restrict__ pos, const double4* __restrict__ box,
    const double* __restrict__ px, const double* __restrict__ py,
    const EdmdPart* __restrict__ part, int n, double t, int extrap, double Lx, double Ly, double dr,
    int nb, int slices, unsigned long long* __restrict__ hist) {
    extern __shared__ unsigned int h[];
    __shared__ double2 stages[PCF_WAVES][64];
    __shared__ uint64_t kept[2][PCF_WAVES], flat[2][PCF_WAVES];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const double rmax = dr * nb;
    const double near2 = rmax * rmax * (1 + 1e-9);
    const float inv = (float)(1 / dr), tol = 1e-6f + 4e-7f * nb;
    for (int b = threadIdx.x; b < nb; b += 64 * PCF_WAVES) h[b] = 0;
    const int tiles = (n + 63) / 64, share = PCF_WAVES * slices;
    auto load = [&](int q) {
        return SORTED ? pos[q] : pcf_position(px, py, part, q, t, extrap, Lx, Ly);
    };
    double2* const stage = stages[wave];
    int buf = 0;
    for (int item = blockIdx.x; item < tiles * slices; item += gridDim.x) {
        const int I = item / slices;
        int turn = wave * slices + (item - I * slices); /* tiles until this wavefront's */
        const int i = I * 64 + lane;
        const double2 a = load(i < n ? i : n - 1);
        double4 bi;
        if (SORTED) bi = box[I];
        for (int J0 = I; J0 < tiles; J0 += 64 * PCF_WAVES, buf ^= 1) {
            const int Jl = J0 + 64 * wave + lane;
            bool keep = Jl < tiles, plain = false;
            if (SORTED && keep) {
                const double4 bj = box[Jl];
                const double ux = pcf_apart(bi.x, bi.y, bj.x, bj.y, Lx);
                const double uy = pcf_apart(bi.z, bi.w, bj.z, bj.w, Ly);
                if (ux * ux + uy * uy > near2 * (1 + 1e-9)) keep = false;
                plain = bj.y - bi.x < Lx / 2 && bj.x - bi.y > -Lx / 2 && bj.w - bi.z < Ly / 2 &&
                        bj.z - bi.w > -Ly / 2;
            }
            const uint64_t k = __ballot(keep), f = __ballot(plain);
            if (lane == 0) {
                kept[buf][wave] = k;
                flat[buf][wave] = f;
            }
            __syncthreads(); /* two buffers: the next round's writes need no other */
            for (int w = 0; w < PCF_WAVES; ++w) {
                uint64_t todo = (uint64_t)uni64((int64_t)kept[buf][w]);
                for (;;) {
                    const int here = __popcll(todo);
                    if (turn >= here) {
                        turn -= here;
                        break;
                    }
                    for (; turn; --turn) todo &= todo - 1;
                    const int at = (int)__builtin_ctzll(todo);
                    todo &= todo - 1;
                    turn = share - 1;
                    const int J = J0 + 64 * w + at;
                    const int j0 = J * 64, jn = n - j0 < 64 ? n - j0 : 64;
                    WAVE_SYNC();
                    stage[lane] = load(lane < jn ? j0 + lane : j0);
                    WAVE_SYNC();
                    const int first = J == I ? lane : -1; /* j > i */
                    if (((uint64_t)uni64((int64_t)flat[buf][w]) >> at) & 1)
                        pcf_tile<false>(stage, jn, a, i < n, first, Lx, Ly, dr, inv, tol, rmax, near2, nb, h);
                    else
                        pcf_tile<true>(stage, jn, a, i < n, first, Lx, Ly, dr, inv, tol, rmax, near2, nb, h);
                }
            }
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nb; b += 64 * PCF_WAVES)
        if (h[b]) atomicAdd(&hist[b], (unsigned long long)h[b]);
}

size_t edmd_pcf_scratch(int n) {
    const size_t tiles = ((size_t)n + 63) / 64;
    return tiles * 64 * (sizeof(double2) + sizeof(int)) + tiles * sizeof(double4) +
           PCF_GRID * PCF_GRID * sizeof(int);
}

hipError_t edmd_launch_pcf_pairs(const double* x, const double* y, const EdmdPart* part, int n,
                                 double t, int extrap, double Lx, double Ly, double dr, int nb,
                                 unsigned long long* hist, void* scratch, hipStream_t s) {
    const int tiles = (n + 63) / 64;
    /* Sorted where the distances counted leave out about half the box and more,
     * the tiles' own size (16 disks' spacings) counted in: below that the
     * tests leave out no tile.  The sort's five launches cost 20 us, all pairs
     * of 2000 disks 25 us, of 4096 about 60. */
    const double reach = 2 * dr * nb, gap = 16 * sqrt(Lx * Ly / n);
    const bool sorted = n >= 4096 && Lx > 0 && Ly > 0 && (reach + gap) * (reach + gap) < 0.6 * Lx * Ly;
    /* two workgroups a CU (60 us at n = 60000, 81 with one); more only so that
     * no LDS count passes 2^32 */
    const double pairs = 0.5 * (double)n * (double)n;
    const int slices = tiles >= 256 ? 1 : (tiles >= 32 ? 2 : 4);
    const long long most = (long long)tiles * slices;
    long long blocks = (long long)ceil(pairs / 2e9);
    blocks = blocks < 512 ? 512 : blocks;
    blocks = blocks > most ? most : blocks;
    const size_t dyn = (size_t)nb * sizeof(unsigned int);
    double2* pos = (double2*)scratch;
    double4* box = (double4*)(pos + (size_t)tiles * 64);
    int* cnt = (int*)(box + tiles);
    int* place = cnt + PCF_GRID * PCF_GRID;
    const int cells = sorted ? PCF_GRID * PCF_GRID : 0, most_clear = nb > cells ? nb : cells;
    const void* f = sorted ? (const void*)k_pcf_pairs<true> : (const void*)k_pcf_pairs<false>;
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 32768 * 4);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k_pcf_clear, dim3((most_clear + 255) / 256), dim3(256), 0, s, hist, nb, cnt,
                       cells);
    if (sorted) {
        hipLaunchKernelGGL(k_pcf_count, dim3((n + 255) / 256), dim3(256), 0, s, x, y, part, n, t,
                           extrap, Lx, Ly, cnt, place);
        hipLaunchKernelGGL(k_pcf_place, dim3((n + PCF_SORT_THREADS - 1) / PCF_SORT_THREADS),
                           dim3(PCF_SORT_THREADS), 0, s, x, y, part, n, t, extrap, Lx, Ly, cnt,
                           place, pos);
        hipLaunchKernelGGL(k_pcf_boxes, dim3((tiles + 3) / 4), dim3(256), 0, s, pos, n, box);
        hipLaunchKernelGGL(k_pcf_pairs<true>, dim3((unsigned)blocks), dim3(64 * PCF_WAVES), dyn, s,
                           pos, box, x, y, part, n, t, extrap, Lx, Ly, dr, nb, slices, hist);
    } else {
        hipLaunchKernelGGL(k_pcf_pairs<false>, dim3((unsigned)blocks), dim3(64 * PCF_WAVES), dyn, s,
                           pos, box, x, y, part, n, t, extrap, Lx, Ly, dr, nb, slices, hist);
    }
    return hipGetLastError();
}
