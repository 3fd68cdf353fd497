// stage.hip -- small transfers between device state and pinned host memory.
//
// A call's results (positions, forces, counts, one replica) and inputs are a few arrays of
// some kilobytes.  A copy each from pageable memory held the stream up for 10 to 20 us; one
// kernel that reads or writes the pinned, device-mapped buffer moves them together in about
// the time of a launch, and the caller copies to or from its own arrays on the host.  Bound by
// the launch and the link.  Reading back 256 replicas of 200 ions took six copies each: with
// their 400 steps 41.4 -> 27.6 ms.  An INTERACT call of 2300 particles 125.6 -> 89.5 us, five steps,
// each with its transfers and energies, of them 1176 -> 962 us.
#include "engine.h"

namespace bromoc {

constexpr int ST_BLOCK = 256;
static dim3 st_grid(int64_t n) {
    const int64_t b = (n + ST_BLOCK - 1) / ST_BLOCK;
    return dim3((unsigned)(b < 1 ? 1 : b > 1024 ? 1024 : b));
}

// double4 positions to x, y, z
__global__ __launch_bounds__(ST_BLOCK) void k_stage_pos_out(const double4 *pos, int n, double *x,
                                                            double *y, double *z) {
    for (int i = blockIdx.x * ST_BLOCK + threadIdx.x; i < n; i += gridDim.x * ST_BLOCK) {
        const double4 p = pos[i];
        x[i] = p.x; y[i] = p.y; z[i] = p.z;
    }
}

// x, y, z, the atnam2 and signed atnam types into both position buffers and the type arrays
__global__ __launch_bounds__(ST_BLOCK) void k_stage_pos_in(const double *x, const double *y,
                                                           const double *z, const int32_t *t2h,
                                                           const int32_t *tyh, int n, double4 *p0,
                                                           double4 *p1, int32_t *t2, int32_t *ty) {
    for (int i = blockIdx.x * ST_BLOCK + threadIdx.x; i < n; i += gridDim.x * ST_BLOCK) {
        const int32_t t = t2h[i];
        const double4 p = make_double4(x[i], y[i], z[i], __hiloint2double(i, t));
        p0[i] = p;
        p1[i] = p;
        t2[i] = t;
        ty[i] = tyh[i];
    }
}

// several arrays of 32-bit words at once, one per block row
__global__ __launch_bounds__(ST_BLOCK) void k_stage_copy(StageCopies c) {
    const int q = blockIdx.y;
    const uint32_t *s = (const uint32_t *)c.src[q];
    uint32_t *d = (uint32_t *)c.dst[q];
    for (int64_t i = blockIdx.x * ST_BLOCK + threadIdx.x; i < c.words[q]; i += (int64_t)gridDim.x * ST_BLOCK)
        d[i] = s[i];
}

// one replica of a batch: its count, energy and buffer counts, then its particles from lo on
__global__ __launch_bounds__(ST_BLOCK) void k_stage_replica(StageReplica a) {
    const int n = a.ntot[a.r], off = a.off[a.r];
    const int t = blockIdx.x * ST_BLOCK + threadIdx.x;
    if (t == 0) { a.o_n[0] = n; a.o_ener[0] = a.gener[a.r]; }
    if (t < a.nbuf) a.o_nat[t] = a.nat[t];
    for (int i = t; i < min(n - a.lo, a.max); i += gridDim.x * ST_BLOCK) {
        const int s = off + a.lo + i;
        const double4 p = a.pos[s];
        a.o_x[i] = p.x; a.o_y[i] = p.y; a.o_z[i] = p.z;
        a.o_ty[i] = a.typei[s];
        a.o_ib[i] = a.ibuffer[s];
    }
}

hipError_t launch_stage_pos_out(const double4 *pos, int n, double *x, double *y, double *z,
                                hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stage_pos_out, st_grid(n), dim3(ST_BLOCK), 0, s, pos, n, x, y, z);
    return hipGetLastError();
}
hipError_t launch_stage_pos_in(const double *x, const double *y, const double *z,
                               const int32_t *t2h, const int32_t *tyh, int n, double4 *p0,
                               double4 *p1, int32_t *t2, int32_t *ty, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_stage_pos_in, st_grid(n), dim3(ST_BLOCK), 0, s, x, y, z, t2h, tyh, n, p0, p1, t2, ty);
    return hipGetLastError();
}
hipError_t launch_stage_copy(const StageCopies &c, hipStream_t s) {
    int64_t m = 0;
    for (int q = 0; q < c.n; q++) m = c.words[q] > m ? c.words[q] : m;
    if (m <= 0) return hipSuccess;
    dim3 g = st_grid(m);
    g.y = (unsigned)c.n;
    hipLaunchKernelGGL(k_stage_copy, g, dim3(ST_BLOCK), 0, s, c);
    return hipGetLastError();
}
hipError_t launch_stage_replica(const StageReplica &a, hipStream_t s) {
    hipLaunchKernelGGL(k_stage_replica, st_grid(a.max > a.nbuf ? a.max : a.nbuf), dim3(ST_BLOCK), 0, s, a);
    return hipGetLastError();
}

}  // namespace bromoc
