// batch.hip -- replica batches: many independent ion systems advanced together.
//
// Every replica owns a contiguous range of particle slots [off, off + cap) in shared
// arrays; the pair tables, the repulsion map and the BD constants are shared, each replica
// has its own static field and GCMC buffers.  One BD step of all replicas is one launch of
// k_batch_step: its wavefronts take (replica, slot) work items -- a fixed table ordered by
// replica size, largest first; a slot beyond the replica's present count is passed over --
// one each (from a device queue where BROMOC_BATCH_BLOCKS asks for it), gather the ion's pair
// forces over its own replica's particles (all pairs, as energy.mono.f90:117-194), its grid
// corners, and apply DYNAMICS0/1/2.  k_batch_noise draws the Gaussians of several steps at
// once.  k_batch_gcmc runs
// GRAND (grand.f90:40-118) for every replica at once, one workgroup per replica, with
// INTERACT energies (interact.f90:19-419, ions only) reduced across the workgroup.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "device.h"

namespace bromoc {

// ---- step and cycle counters: before GRAND (gcmc), or before `steps` BD steps whose noise
// follows (ctl[4]: the counter of the first of them); and the queue counter of one step
__global__ void k_batch_prep(BatchParams B, int gcmc, int steps) {
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    if (gcmc) {
        B.ctl[5] = B.ctl[6] + B.ctl[2];
        B.ctl[2] += 1;
    } else {
        B.ctl[4] = B.ctl[1] + B.ctl[0];
        B.ctl[0] += steps;
    }
}
__global__ void k_batch_queue(int32_t *queue) {
    if (threadIdx.x == 0 && blockIdx.x == 0) queue[0] = 0;
}

hipError_t launch_batch_prep(const BatchParams &b, int gcmc, int steps, hipStream_t s) {
    hipLaunchKernelGGL(k_batch_prep, dim3(1), dim3(64), 0, s, b, gcmc, steps);
    return hipGetLastError();
}

// The Gaussians of `steps` steps from the counter ctl[4], row per step, three per item: one
// thread per item and step.  Drawn in the step kernel they took every lane of a wavefront for
// the three that need one (a tenth of a step at 4000 ions a replica, a third at 200).
__global__ __launch_bounds__(BLOCK) void k_batch_noise(BatchParams B, int steps) {
    const int w = blockIdx.x * BLOCK + threadIdx.x;
    if (w >= B.nitems) return;
    const int2 it = B.items[w];   // replica, slot in it
    if (it.y >= B.ntot[it.x]) return;
    const int row = blockIdx.y;
    double g[3];
    philox_gauss3((uint64_t)B.ctl[3], (uint64_t)B.ctl[4] + row, (uint64_t)it.x, it.y, g);
    double *o = B.noise + 3 * ((size_t)row * B.nitems + w);
    o[0] = g[0]; o[1] = g[1]; o[2] = g[2];
}

hipError_t launch_batch_noise(const BatchParams &b, int steps, hipStream_t s) {
    if (b.nitems <= 0 || steps <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_batch_noise, dim3((b.nitems + BLOCK - 1) / BLOCK, steps), dim3(BLOCK), 0, s, b, steps);
    return hipGetLastError();
}

// ---- one BD step (or ENERGY) of every replica
// G lanes per target: each wavefront holds 64/G targets, every lane group of G lanes takes
// its own work item (a moving ion of some replica), strides over that replica's particles
// and reduces its sums within the group.  Small replicas want small groups (more targets
// in flight, the per-item latencies overlap); the autotuner picks G.
//
// A lane evaluates the analytic tail of 32 partners straight through, leaving out the pairs
// within table range and noting each as a bit, then works the bits off.  With a branch to the
// table per pair a wavefront took it at most iterations for the 2 % of its lanes that have a
// pair in range (some other replica's or part of the box in each lane), and waited for the
// knots each time.  The grid corners are loaded before the pair loop and used after it.
// Measured per step, before and after (with the noise drawn beforehand, and no prefix kernel):
// 256 replicas of 100..4000 ions 1.79 -> 0.86 ms, 256 replicas of 200 ions 101 -> 53 us.
// feature bits of the k_batch_step specialisations
constexpr int BF_PHIX = 1;       // static field grids
constexpr int BF_PHIV = 2;       // repulsion map
constexpr int BF_ANALYTIC = 4;   // some pair type is analytic (else every pair is tabulated)

template <int G>
__device__ __forceinline__ double group_sum(double v) {
#pragma unroll
    for (int off = 16; off < G; off <<= 1) v += __shfl_xor(v, off, WAVE);
    return G == 8 ? half_row_sum(v) : row_sum(v);
}

template <int FEAT, int G>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu((FEAT & BF_ANALYTIC) ? 2 : 4)))
void k_batch_step(BatchParams B) {
    static_assert(G >= 8 && G <= WAVE && (WAVE % G) == 0, "lane group");
    constexpr bool ANA = (FEAT & BF_ANALYTIC) != 0;
    const StepParams &P = B.sp;
    // every (target type, partner type) row of the shared tables
    extern __shared__ double4 s_dyn[];
    const int nt1 = P.nttyp + 1, nrow = nt1 * nt1;
    DevPair *s_rows = reinterpret_cast<DevPair *>(s_dyn);
    double4 *s_tail = s_dyn + (size_t)nrow * (sizeof(DevPair) / sizeof(double4));
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wv = tid >> 6;
    const int sub = lane / G, sl = lane % G;
    for (int k = tid; k < nrow; k += BLOCK) {
        const DevPair d = P.rows[k];
        s_rows[k] = d;
        s_tail[k] = make_double4(d.sc3, d.fct, ANA && !(d.flags & PF_EFPOT) ? -1.0 : d.dm2hi, 0.0);
    }
    __syncthreads();
    const bool nonbond = (P.flags & QNONBOND) && (P.flags & QPAR);
    int next = (blockIdx.x * WPB + wv) * (WAVE / G) + sub;
    for (;;) {
        int w;
        if (B.persistent) {
            int v = 0;
            if (sl == 0) v = atomicAdd(&B.queue[0], 1);
            w = __shfl(v, sub * G, WAVE);
        } else {
            w = next;
            next = INT_MAX;
        }
        if (w >= B.nitems) break;
        const int2 it = B.items[w];
        const int r = it.x, t = it.y;
        const int off = B.off[r], n = B.ntot[r];
        if (t >= n) continue;   // no particle in this slot now
        const double4 *const pos = B.pos + off;
        const double4 pa = pos[t];
        const int itype = abs(B.typei[off + t]);
        const int t2 = __double2loint(pa.w);
        const DevPair *rowp = s_rows + t2 * nt1;
        const double4 *tailp = s_tail + t2 * nt1;
        // grid corners: lanes 0..7 of the group (staticf1.f90:45-118, vdwgd1trln.f90:50-161)
        bool okx = false, okv = false;
        double xx = 0.0, xy = 0.0, xz = 0.0, vx = 0.0, vy = 0.0, vz = 0.0;
        int xi = 0, xj = 0, xk = 0, vi = 0, vj = 0, vk = 0;
        float phx = 0.0f;
        int8_t phv = 0;
        if constexpr ((FEAT & BF_PHIX) != 0) {
            const GridGeom &g = P.gx;
            okx = pa.x <= g.xbcen + g.tranx && pa.x >= g.xbcen - g.tranx &&
                  pa.y <= g.ybcen + g.trany && pa.y >= g.ybcen - g.trany &&
                  pa.z <= g.zbcen + g.tranz && pa.z >= g.zbcen - g.tranz;
            if (okx && sl < 8) {
                grid_cell(g, pa.x, pa.y, pa.z, xx, xy, xz, xi, xj, xk);
                phx = B.phix[r][tri_node(g, xi, xj, xk, sl)];
            }
        }
        if constexpr ((FEAT & BF_PHIV) != 0) {
            const GridGeom &g = P.gv;
            okv = pa.x <= g.xbcen + g.tranx && pa.x >= g.xbcen - g.tranx &&
                  pa.y <= g.ybcen + g.trany && pa.y >= g.ybcen - g.trany &&
                  pa.z <= P.vzmax && pa.z >= P.vzmin;
            if (okv && sl < 8) {
                grid_cell(g, pa.x, pa.y, pa.z, vx, vy, vz, vi, vj, vk);
                phv = P.phiv[tri_node(g, vi, vj, vk, sl)];
            }
        }
        double gk[3] = {0.0, 0.0, 0.0};   // Gaussians of the update
        if (B.mode == 1 && sl == 0) {
            const double *nr = B.noise + 3 * ((size_t)B.noise_row * B.nitems + w);
            gk[0] = nr[0]; gk[1] = nr[1]; gk[2] = nr[2];
        }
        double fx = 0.0, fy = 0.0, fz = 0.0, et = 0.0, eel = 0.0, evd = 0.0, esr = 0.0;
        auto pair_loop = [&](auto en) {
            constexpr bool EN = decltype(en)::value;
            constexpr int PU = 2;   // one: 1.00 ms, four: 1.00 ms (registers) against 0.86
            for (int base = sl; base < n; base += 32 * G) {
                uint32_t m = 0u;
                const int cnt = min(32, (n - base + G - 1) / G);
                // PU partners per iteration: their loads and chains overlap
#pragma unroll 1
                for (int k0 = 0; k0 < cnt; k0 += PU) {
                    double4 q[PU];
#pragma unroll
                    for (int u = 0; u < PU; u++) q[u] = pos[min(base + (k0 + u) * G, n - 1)];
#pragma unroll
                    for (int u = 0; u < PU; u++) {
                        const int p = base + (k0 + u) * G;
                        const bool on = p < n && p != t;
                        const int tj = __double2loint(q[u].w);
                        const double4 tl = tailp[tj];
                        const double dx = pa.x - q[u].x, dy = pa.y - q[u].y, dz = pa.z - q[u].z;
                        const double d2 = on ? pair_d2(dx, dy, dz) : 1e30;
                        double f;
                        if (ANA && tl.z < 0.0) {
                            double q0 = 0.0, q1 = 0.0, q2 = 0.0;
                            f = pair_analytic(rowp[tj], P, d2, q0, q1, q2);
                            f = on ? f : 0.0;
                            if constexpr (EN) {
                                // an ion pair's energy is counted by its higher-index ion
                                // (energy.mono.f90:117)
                                const bool ce = on && p < t;
                                eel += ce ? q0 : 0.0;
                                evd += ce ? q1 : 0.0;
                                esr += ce ? q2 : 0.0;
                            }
                        } else {
                            const double ri = rsqrt_s26(d2), i2 = ri * ri, c = tl.x * (i2 * i2 * i2);
                            const double fr = tl.y * ri;
                            const bool near = d2 <= tl.z;   // false for a masked pair
                            f = (6.0 * c + fr) * i2;
                            f = on && !near ? f : 0.0;
                            if constexpr (EN) et += on && !near && p < t ? c + fr : 0.0;
                            m |= near ? 1u << (k0 + u) : 0u;
                        }
                        fx = fma(f, dx, fx);
                        fy = fma(f, dy, fy);
                        fz = fma(f, dz, fz);
                    }
                }
                while (m) {   // the pairs within table range
                    const int k = __ffs(m) - 1, p = base + k * G;
                    m &= m - 1u;
                    const double4 q = pos[p];
                    const DevPair &row = rowp[__double2loint(q.w)];
                    const double dx = pa.x - q.x, dy = pa.y - q.y, dz = pa.z - q.z;
                    const double d2 = pair_d2(dx, dy, dz), ri = rsqrt_s26(d2);
                    double y;
                    const double f = pair_table(row, P.ep, P.ires, d2, ri, y);
                    if constexpr (EN) et += p < t ? y : 0.0;
                    fx = fma(f, dx, fx);
                    fy = fma(f, dy, fy);
                    fz = fma(f, dz, fz);
                }
            }
        };
        if (nonbond) {
            if (B.write_energy) pair_loop(std::true_type{});
            else pair_loop(std::false_type{});
        }
        double egx = 0.0, egv = 0.0;
        bool warned = false;
        if constexpr ((FEAT & BF_PHIX) != 0) {
            if (okx && sl < 8)
                tri_apply(P.gx, (double)phx, xx, xy, xz, xi, xj, xk, sl, P.celec * P.cg[itype], fx, fy, fz, egx);
        }
        if constexpr ((FEAT & BF_PHIV) != 0) {
            double ph = 0.0;
            if (okv && sl < 8) {
                ph = (double)phv;
                double esvdw = P.svdw;
                if (P.flags & QSVDW) esvdw = P.svdw * P.scal[t2];
                tri_apply(P.gv, ph, vx, vy, vz, vi, vj, vk, sl, esvdw, fx, fy, fz, egv);
            }
            warned = okv && half_row_sum(ph) >= P.thold8;   // integers: exact
        }
        fx = group_sum<G>(fx);
        fy = group_sum<G>(fy);
        fz = group_sum<G>(fz);
        if (B.write_energy) {
            et = group_sum<G>(et);
            eel = group_sum<G>(eel);
            evd = group_sum<G>(evd);
            esr = group_sum<G>(esr);
            egx = group_sum<G>(egx);
            egv = group_sum<G>(egv);
        }
        if (sl == 0) {
            const int64_t i = off + t;
            if (warned) atomicAdd(&B.warn[(size_t)r * B.warn_stride + t2], 1);
            if (B.write_energy) {
                double *ep_ = B.epart + i;
                const int64_t cs = B.ecap;
                ep_[E_GSBPA * cs] = egx;
                ep_[E_VDWGD * cs] = egv;
                ep_[E_EFPOT * cs] = et;
                ep_[E_ELEC * cs] = eel;
                ep_[E_VDW * cs] = evd;
                ep_[E_SRPMF * cs] = esr;
            }
            if (B.write_forces) {
                B.fx[i] = fx;
                B.fy[i] = fy;
                B.fz[i] = fz;
            }
            if (B.mode == 1) {
                const double F[3] = {fx, fy, fz};
                B.poso[i] = bd_move(P, false, itype, pa, F, gk,
                                    B.nfwd + (size_t)r * B.flux_stride,
                                    B.nbwd + (size_t)r * B.flux_stride);
            }
        }
    }
}

template <int FEAT>
static void launch_batch_feat(const BatchParams &q, int lanes, dim3 grid, size_t lds,
                              hipStream_t s) {
    if (lanes == 8)
        hipLaunchKernelGGL((k_batch_step<FEAT, 8>), grid, dim3(BLOCK), lds, s, q);
    else if (lanes == 16)
        hipLaunchKernelGGL((k_batch_step<FEAT, 16>), grid, dim3(BLOCK), lds, s, q);
    else if (lanes == 32)
        hipLaunchKernelGGL((k_batch_step<FEAT, 32>), grid, dim3(BLOCK), lds, s, q);
    else
        hipLaunchKernelGGL((k_batch_step<FEAT, 64>), grid, dim3(BLOCK), lds, s, q);
}

hipError_t launch_batch_step(const BatchParams &b, int blocks, int lanes, hipStream_t s) {
    int feat = 0;
    if (b.sp.flags & QPHIX) feat |= BF_PHIX;
    if (b.sp.flags & QPHIV) feat |= BF_PHIV;
    if (!b.sp.all_efpot) feat |= BF_ANALYTIC;
    if (lanes != 8 && lanes != 16 && lanes != 32) lanes = 64;
    BatchParams q = b;
    q.persistent = blocks > 0 ? 1 : 0;
    const int per_block = WPB * (WAVE / lanes);
    dim3 grid(blocks > 0 ? blocks : std::max(1, (b.nitems + per_block - 1) / per_block));
    const int nt1 = b.sp.nttyp + 1;
    const size_t lds = (size_t)nt1 * nt1 * (sizeof(DevPair) + sizeof(double4));
    if (q.persistent) hipLaunchKernelGGL(k_batch_queue, dim3(1), dim3(64), 0, s, q.queue);
    switch (feat) {
        case 0: launch_batch_feat<0>(q, lanes, grid, lds, s); break;
        case 1: launch_batch_feat<1>(q, lanes, grid, lds, s); break;
        case 2: launch_batch_feat<2>(q, lanes, grid, lds, s); break;
        case 3: launch_batch_feat<3>(q, lanes, grid, lds, s); break;
        case 4: launch_batch_feat<4>(q, lanes, grid, lds, s); break;
        case 5: launch_batch_feat<5>(q, lanes, grid, lds, s); break;
        case 6: launch_batch_feat<6>(q, lanes, grid, lds, s); break;
        default: launch_batch_feat<7>(q, lanes, grid, lds, s); break;
    }
    return hipGetLastError();
}

// ---- GRAND of every replica: one workgroup per replica, attempts in order
// uniform k of replica r in GCMC cycle c: word k%4 of Philox(c, k/4, r, 1; seed, 0)
__device__ __forceinline__ double gcmc_uniform(uint64_t seed, uint64_t cycle, int r, uint64_t k) {
    uint64_t c[4] = {cycle, k >> 2, (uint64_t)r, 1};
    philox4x64(c, seed, 0);
    return (double)(c[k & 3] >> 11) * (1.0 / 9007199254740992.0);
}

// INTERACT of an ion of atnam type jtype at (xj, yj, zj) in replica r, as particle j (j ==
// ntot: an insertion trial): grids, then every other ion (interact.f90:155-204).  All
// threads of the block call it; the sum is returned to thread 0.
__device__ double batch_interact(const BatchParams &B, int r, int off, int ntot, double xj,
                                 double yj, double zj, int jtype, int j, bool alert,
                                 double *s_red) {
    const StepParams &P = B.sp;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1);
    const int nt1 = P.nttyp + 1;
    const int jt2 = P.nwtype[jtype];
    double e = 0.0;
    if (tid < WAVE) {
        bool wall = false;
        const double eg = interact_grids(P, B.phix[r], true, P.cg[jtype], xj, yj, zj, jt2, wall);
        if (tid == 0) {
            e += eg;
            if (wall && alert) atomicAdd(&B.warn[(size_t)r * B.warn_stride + jt2], 1);
        }
    }
    if (P.flags & QNONBOND) {
        for (int i = tid; i < ntot; i += BLOCK) {
            if (i == j) continue;
            const double4 q = B.posw[off + i];
            const double dx = q.x - xj, dy = q.y - yj, dz = q.z - zj;
            const double d2 = dx * dx + dy * dy + dz * dz;
            const DevPair &pp = P.rows[jt2 * nt1 + __double2loint(q.w)];
            e += (pp.flags & PF_EFPOT) ? gety(pp, P.ep, P.ires, d2) : interact_analytic(pp, P, d2);
        }
    }
    e = wave_sum(e);
    if (lane == 0) s_red[tid >> 6] = e;
    __syncthreads();
    double t = 0.0;
    if (tid == 0)
        for (int k = 0; k < WPB; k++) t += s_red[k];
    __syncthreads();
    return t;
}

__global__ __launch_bounds__(BLOCK) void k_batch_gcmc(BatchParams B) {
    const StepParams &P = B.sp;
    const int r = blockIdx.x;
    const int nb = B.nbuf[r];
    if (nb <= 0 || B.ngcmc <= 0) return;
    __shared__ double s_red[WPB];
    __shared__ double s_d[4];
    __shared__ int s_i[8];
    __shared__ int s_cnt[WPB];
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wv = tid >> 6;
    const int off = B.off[r], cap = B.cap[r], nf = B.nfix[r];
    const size_t gb = (size_t)r * B.gstride;
    const int32_t *ibfftyp = B.ibfftyp + gb, *ntotat = B.ntotat + gb;
    const double *avnum = B.avnum + gb, *mu = B.mu + gb, *kb = B.kb + gb;
    const double *lzmin = B.lzmin + gb, *lzmax = B.lzmax + gb;
    const int8_t *bias = B.bias + gb;
    int32_t *nat = B.nat + gb;
    int32_t *prob = B.prob + B.probofs[r];
    const double *bx = B.gbox + 6 * (size_t)r;
    const double lx = bx[0], ly = bx[1], cx = bx[2], cy = bx[3], cz = bx[4], ikbt = bx[5];
    const uint64_t seed = (uint64_t)B.ctl[3], cycle = (uint64_t)B.ctl[5];
    const int64_t icycle = (int64_t)cycle + 1;
    const double nbufferr = (double)nb;
    int ntot = B.ntot[r];
    uint64_t k = 0;       // uniforms drawn (thread 0)
    double ener = B.gener[r];
    for (int ig = 0; ig < B.ngcmc; ig++) {
        // ---- the trial (grand.f90:42-50, 77-84), drawn by thread 0
        if (tid == 0) {
            int mode = 0, ib = 0, ip = 0, itype = 0;
            double xn = 0.0, yn = 0.0, zn = 0.0;
            if (gcmc_uniform(seed, cycle, r, k++) < 0.5) {
                ib = (int)(nbufferr * gcmc_uniform(seed, cycle, r, k++)) + 1;
                if (ib <= nb && avnum[ib] > 0.0) {
                    mode = 1;
                    itype = ibfftyp[ib];
                    xn = lx * (gcmc_uniform(seed, cycle, r, k++) - 0.5) + cx;
                    yn = ly * (gcmc_uniform(seed, cycle, r, k++) - 0.5) + cy;
                    zn = lzmin[ib] + (lzmax[ib] - lzmin[ib]) * gcmc_uniform(seed, cycle, r, k++);
                }
            } else {
                ib = (int)(nbufferr * gcmc_uniform(seed, cycle, r, k++)) + 1;
                const double natib = ib <= nb ? (double)nat[ib] : 0.0;
                ip = (int)(natib * gcmc_uniform(seed, cycle, r, k++)) + 1;
                if (ib <= nb && ip <= nat[ib]) {
                    mode = 2;
                    itype = ibfftyp[ib];
                }
            }
            s_i[0] = mode; s_i[1] = ib; s_i[2] = ip; s_i[3] = itype; s_i[4] = -1;
            s_d[0] = xn; s_d[1] = yn; s_d[2] = zn;
        }
        __syncthreads();
        const int mode = s_i[0], ib = s_i[1], ip = s_i[2], itype = s_i[3];
        if (mode == 2) {
            // FIND (find.f90:26-32): the ip-th moving ion of buffer ib, in slot order
            int seen = 0;
            for (int c0 = nf; c0 < ntot && seen < ip; c0 += BLOCK) {
                const int a = c0 + tid;
                const bool hit = a < ntot && B.ibuffer[off + a] == ib;
                const uint64_t m = __ballot(hit);
                if (lane == 0) s_cnt[wv] = __popcll(m);
                __syncthreads();
                int before = seen;
                for (int q = 0; q < wv; q++) before += s_cnt[q];
                const int rank = before + __popcll(m & ((1ull << lane) - 1ull)) + 1;
                if (hit && rank == ip) s_i[4] = a;
                int tot = 0;
                for (int q = 0; q < WPB; q++) tot += s_cnt[q];
                __syncthreads();
                seen += tot;
            }
            __syncthreads();
            if (tid == 0 && s_i[4] >= 0) {
                const double4 q = B.posw[off + s_i[4]];
                s_d[0] = q.x; s_d[1] = q.y; s_d[2] = q.z;
            }
            __syncthreads();
            if (s_i[4] < 0) {   // nat out of step with ibuffer: stop this replica's GRAND
                if (tid == 0) atomicOr(&B.queue[1], 2);
                break;
            }
        }
        if (mode != 0) {
            const int j = mode == 1 ? ntot : s_i[4];
            const double dener = batch_interact(B, r, off, ntot, s_d[0], s_d[1], s_d[2], itype, j,
                                                mode == 2, s_red);
            if (tid == 0) {
                double rate;
                const double natv = mode == 1 ? (double)(nat[ib] + 1) : (double)nat[ib];
                if (bias[ib]) {
                    rate = (avnum[ib] + kb[ib] * (avnum[ib] - (double)(ntotat[ib] / icycle)));
                    rate = rate * exp(-(dener - mu[ib]) * ikbt) / natv;
                } else {
                    rate = mode == 1 ? (avnum[ib] / (nat[ib] + 1)) * exp(-(dener - mu[ib]) * ikbt)
                                     : (avnum[ib] / nat[ib]) * exp(-(dener - mu[ib]) * ikbt);
                }
                rate = mode == 1 ? rate / (1.0 + rate) : 1.0 / (1.0 + rate);
                int nt_new = ntot;
                if (gcmc_uniform(seed, cycle, r, k++) <= rate) {
                    if (mode == 1) {
                        if (ntot + 1 > cap) {
                            atomicOr(&B.queue[1], 1);
                            nt_new = -1;
                        } else {
                            ener = ener + dener;
                            nat[ib] = nat[ib] + 1;
                            const int a = ntot;
                            const int t2 = P.nwtype[itype];
                            B.posw[off + a] = make_double4(s_d[0], s_d[1], s_d[2],
                                                           __hiloint2double(0, t2));
                            B.typei[off + a] = s_d[2] < cz ? -itype : itype;
                            B.ibuffer[off + a] = ib;
                            nt_new = ntot + 1;
                        }
                    } else {
                        ener = ener - dener;
                        const int a = s_i[4], last = ntot - 1;
                        B.posw[off + a] = B.posw[off + last];
                        B.typei[off + a] = B.typei[off + last];
                        B.ibuffer[off + a] = B.ibuffer[off + last];
                        nat[ib] = nat[ib] - 1;
                        nt_new = ntot - 1;
                    }
                }
                s_i[5] = nt_new;
            }
            __syncthreads();
            if (s_i[5] < 0) break;   // capacity exceeded
            ntot = s_i[5];
        }
        if (tid == 0)
            for (int b = 1; b <= nb; b++) prob[(size_t)(b - 1) * (cap + 1) + nat[b]] += 1;
        __syncthreads();
    }
    if (tid == 0) {
        B.ntot[r] = ntot;
        B.gener[r] = ener;
    }
}

hipError_t launch_batch_gcmc(const BatchParams &b, hipStream_t s) {
    hipLaunchKernelGGL(k_batch_gcmc, dim3(b.nrep), dim3(BLOCK), 0, s, b);
    return hipGetLastError();
}

// ---- energies of every replica: one block per replica, fixed-order tree per category
__global__ __launch_bounds__(BLOCK) void k_batch_reduce(BatchParams B, double *out) {
    __shared__ double s[BLOCK];
    const int r = blockIdx.x, tid = threadIdx.x;
    const int off = B.off[r], n = B.ntot[r];
    for (int cat = 0; cat < NE; cat++) {
        const double *src = B.epart + (size_t)cat * B.ecap + off;
        double acc = 0.0;
        for (int k = tid; k < n; k += BLOCK) acc += src[k];
        s[tid] = acc;
        __syncthreads();
        for (int h = BLOCK / 2; h > 0; h >>= 1) {
            if (tid < h) s[tid] += s[tid + h];
            __syncthreads();
        }
        if (tid == 0) out[(size_t)r * NE + cat] = s[0];
        __syncthreads();
    }
}

hipError_t launch_batch_reduce(const BatchParams &b, double *out, hipStream_t s) {
    hipLaunchKernelGGL(k_batch_reduce, dim3(b.nrep), dim3(BLOCK), 0, s, b, out);
    return hipGetLastError();
}

}  // namespace bromoc

// ======================================================================= host side
using namespace bromoc;

namespace {

constexpr int BATCH_GRAPH_K = 32;   // steps per captured graph without GCMC
// steps whose noise is drawn by one launch, within a bounded buffer
constexpr int BATCH_NOISE_ROWS = 16;
constexpr size_t BATCH_NOISE_BYTES = size_t(256) << 20;
// slots of a replica that bromoc_batch_get stages at a time (1 MiB of pinned memory)
constexpr size_t BATCH_GET_SLOTS = 32768;

template <typename T>
hipError_t balloc(std::vector<void *> &al, T **p, size_t n) {
    void *q = nullptr;
    hipError_t e = hipMalloc(&q, std::max<size_t>(n, 1) * sizeof(T));
    if (e != hipSuccess) return e;
    al.push_back(q);
    *p = (T *)q;
    return hipMemset(q, 0, std::max<size_t>(n, 1) * sizeof(T));
}

template <typename T>
hipError_t bupload(std::vector<void *> &al, T **p, const T *src, size_t n) {
    hipError_t e = balloc(al, p, n);
    if (e != hipSuccess || !src || n == 0) return e;
    return hipMemcpy(*p, src, n * sizeof(T), hipMemcpyHostToDevice);
}

double pack_t2(int32_t t2) {
    uint64_t bits = (uint64_t)(uint32_t)t2;
    double d;
    std::memcpy(&d, &bits, sizeof(d));
    return d;
}

}  // namespace

struct bromoc_batch {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string err;
    bromoc_ctx *shared = nullptr;
    bromoc_system sys{};
    int nrep = 0, gstride = 1, flux_stride = 1, warn_stride = 1;
    int64_t total = 0;
    std::vector<int32_t> h_off, h_cap, h_nfix, h_nbuf;
    std::vector<int64_t> h_probofs;
    std::vector<void *> allocs;
    BatchParams base{};
    double4 *pos[2] = {nullptr, nullptr};
    int cur = 0;
    int32_t *warn_scratch = nullptr;
    double *ered = nullptr;
    int blocks = -1;   // autotuned launch shape (0: one item per lane group, no queue)
    int lanes = 64;    // lanes per target
    int noise_rows = 1;   // steps the noise buffer holds
    void *pin = nullptr;  // pinned staging of bromoc_batch_get
    size_t pin_cap = 0;
    int64_t h_ctl[8] = {};
    struct Graph {
        hipGraphExec_t exec = nullptr;
        int len = -1, gcmc = -1, ngcmc = -1, blocks = -1, lanes = -1;
    } graph[2];
};

namespace {

int bfail(bromoc_batch *b, int code, const std::string &m) {
    if (b) b->err = m;
    return code;
}

#define BCHK(b, expr)                                                                      \
    do {                                                                                   \
        hipError_t e_ = (expr);                                                            \
        if (e_ != hipSuccess)                                                              \
            return bfail((b), BROMOC_E_HIP, std::string(#expr ": ") + hipGetErrorString(e_)); \
    } while (0)

BatchParams params_now(bromoc_batch *b) {
    BatchParams p = b->base;
    p.pos = b->pos[b->cur];
    p.poso = b->pos[b->cur ^ 1];
    p.posw = b->pos[b->cur];
    return p;
}

// energy.mono.f90:83-110,689 for an ion-only system (no membrane, no reaction fields)
void batch_energies(const double *r, bromoc_energies *out) {
    bromoc_energies E;
    std::memset(&E, 0, sizeof(E));
    double *f = &E.eelec;
    for (int k = 0; k < NE; k++) f[k] = r[k];
    E.ener = E.ememb;
    E.ener = E.ener + E.egsbpa;
    E.ener = E.ener + E.evdwgd;
    E.ener = E.ener + E.eelec + E.evdw + E.esrpmf + E.esrpmfmx + E.ebond + E.eang + E.edihe +
             E.estack + E.ebp + E.eex + E.eqq + E.esolv + E.eqqmx + E.evdwmx + E.eefpot +
             E.eefpotmx + E.econ;
    *out = E;
}

// the counters and noise of the next n <= BATCH_NOISE_ROWS steps
hipError_t enqueue_batch_noise(const BatchParams &p, int n, hipStream_t s) {
    hipError_t e = launch_batch_prep(p, 0, n, s);
    if (e != hipSuccess) return e;
    return launch_batch_noise(p, n, s);
}

hipError_t enqueue_batch_gcmc(const BatchParams &p, hipStream_t s) {
    hipError_t e = launch_batch_prep(p, 1, 0, s);
    if (e != hipSuccess) return e;
    return launch_batch_gcmc(p, s);
}

int batch_sync(bromoc_batch *b) {
    hipError_t e = hipStreamSynchronize(b->stream);
    if (e != hipSuccess) return bfail(b, BROMOC_E_HIP, std::string("kernel: ") + hipGetErrorString(e));
    return BROMOC_OK;
}

// Autotuner: 8, 16, 32 or 64 lanes per target, one work item per lane group, timed on
// ENERGY-only launches whose warnings go to a scratch counter, the best of two rounds (the first
// launches of a process run slow).  The queue is not among the candidates: its persistent
// workgroups take twice the time (256 replicas of 100..4000 ions 2.0 ms against 0.86, of 200
// ions 200 us against 53), since the hardware hands out blocks in the same largest-first order.
// BROMOC_BATCH_BLOCKS and BROMOC_BATCH_LANES force a shape (blocks 0: no queue).
int batch_autotune(bromoc_batch *b) {
    if (b->blocks >= 0) return BROMOC_OK;
    const char *eb = std::getenv("BROMOC_BATCH_BLOCKS"), *el = std::getenv("BROMOC_BATCH_LANES");
    if (eb || el) {
        b->blocks = eb ? std::max(0, std::atoi(eb)) : 0;
        b->lanes = el ? std::atoi(el) : 64;
        if (b->lanes != 8 && b->lanes != 16 && b->lanes != 32) b->lanes = 64;
        return BROMOC_OK;
    }
    const int cl[4] = {8, 16, 32, 64};
    hipEvent_t e0, e1;
    BCHK(b, hipEventCreate(&e0));
    BCHK(b, hipEventCreate(&e1));
    double best = 1e300;
    int pick = 64;
    for (int round = 0; round < 2; round++) {
        for (int l : cl) {
            BatchParams p = params_now(b);
            p.mode = 0;
            p.write_energy = 0;
            p.write_forces = 0;
            p.warn = b->warn_scratch;
            BCHK(b, launch_batch_step(p, 0, l, b->stream));
            BCHK(b, hipEventRecord(e0, b->stream));
            for (int r = 0; r < 3; r++) BCHK(b, launch_batch_step(p, 0, l, b->stream));
            BCHK(b, hipEventRecord(e1, b->stream));
            int st = batch_sync(b);
            if (st) return st;
            float ms = 0.f;
            BCHK(b, hipEventElapsedTime(&ms, e0, e1));
            if (ms < best) { best = ms; pick = l; }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    b->blocks = 0;
    b->lanes = pick;
    return BROMOC_OK;
}

int batch_check_flags(bromoc_batch *b) {
    int32_t q[2] = {0, 0};
    BCHK(b, hipMemcpy(q, b->base.queue, sizeof(q), hipMemcpyDeviceToHost));
    if (q[1] & 1) return bfail(b, BROMOC_E_CAPACITY, "a replica exceeded its capacity in GRAND");
    if (q[1] & 2) return bfail(b, BROMOC_E_STATE, "nat does not match ibuffer in GRAND");
    return BROMOC_OK;
}

}  // namespace

extern "C" {

const char *bromoc_batch_last_error(const bromoc_batch *b) { return b ? b->err.c_str() : "null batch"; }

int bromoc_batch_destroy(bromoc_batch *b) {
    if (!b) return BROMOC_OK;
    (void)hipSetDevice(b->device);
    if (b->stream) (void)hipStreamSynchronize(b->stream);
    for (auto &g : b->graph)
        if (g.exec) (void)hipGraphExecDestroy(g.exec);
    for (void *p : b->allocs) (void)hipFree(p);
    if (b->pin) (void)hipHostFree(b->pin);
    if (b->shared) bromoc_destroy(b->shared);
    if (b->stream) (void)hipStreamDestroy(b->stream);
    delete b;
    return BROMOC_OK;
}

int bromoc_batch_create(const bromoc_system *s, int32_t nrep, const bromoc_replica *reps,
                        int device, bromoc_batch **out) {
    if (!s || !reps || !out || nrep < 1 || nrep > (1 << 16)) return BROMOC_E_ARG;
    *out = nullptr;
    // the replica kernels implement pairs, the trilinear grids and DYNAMICS0/1/2 only
    const uint32_t unsupported = BROMOC_QNUCL | BROMOC_QRFPAR | BROMOC_QRFPSIN | BROMOC_QDNAFREE |
                                 BROMOC_QMEMB | BROMOC_QBSPLINE | BROMOC_QMMIJ | BROMOC_QNMCDEN |
                                 BROMOC_QSPHERE | BROMOC_QECYL;
    if (s->flags & unsupported) {
        fprintf(stderr, "bromoc_batch_create: replicas are ion-only boxes (no CG-DNA, RFPAR, "
                        "MMIJ, membrane, B-spline, per-species map or curved system)\n");
        return BROMOC_E_UNSUPPORTED;
    }
    if (s->nsites != 0 || !(s->flags & BROMOC_QPAR)) return BROMOC_E_ARG;
    const bool qphix = (s->flags & BROMOC_QPHIX) != 0;
    int64_t total = 0;
    int gmax = 0;
    for (int r = 0; r < nrep; r++) {
        const bromoc_replica &R = reps[r];
        if (R.ntot < 0 || R.nfix < 0 || R.nfix > R.ntot || R.capacity < R.ntot ||
            R.capacity < 1 || R.capacity > (1 << 22))
            return BROMOC_E_ARG;
        if (R.ntot > 0 && (!R.x || !R.y || !R.z || !R.typei)) return BROMOC_E_ARG;
        if (qphix && !R.phix) return BROMOC_E_ARG;
        for (int i = 0; i < R.ntot; i++) {
            const int t = std::abs(R.typei[i]);
            if (t <= s->nold || t > s->ntype) return BROMOC_E_ARG;
        }
        if (R.gcmc) {
            const bromoc_gcmc &G = *R.gcmc;
            if (G.nbuffer < 0 || G.nbuffer > 64) return BROMOC_E_ARG;
            if (G.nbuffer > 0 && (!G.ibfftyp || !G.avnum || !G.mu || !G.kb || !G.lzmin ||
                                  !G.lzmax || !G.bufferbias || !G.ntotat || !R.nat ||
                                  (R.ntot > 0 && !R.ibuffer)))
                return BROMOC_E_ARG;
            std::vector<int> cnt(G.nbuffer + 1, 0);
            for (int b = 1; b <= G.nbuffer; b++)
                if (G.ibfftyp[b] <= s->nold || G.ibfftyp[b] > s->ntype) return BROMOC_E_ARG;
            for (int i = 0; i < R.ntot; i++) {
                const int v = R.ibuffer[i];
                if (v < 0 || v > G.nbuffer || (v > 0 && i < R.nfix)) return BROMOC_E_ARG;
                cnt[v]++;
            }
            for (int b = 1; b <= G.nbuffer; b++)
                if (R.nat[b] != cnt[b]) return BROMOC_E_ARG;
            gmax = std::max(gmax, G.nbuffer);
        }
        total += R.capacity;
    }
    if (total > ((int64_t)1 << 27)) return BROMOC_E_ARG;
    // the shared tables through a particle-less single-system context
    bromoc_system sh = *s;
    sh.ntot = 0;
    sh.nfix = 0;
    sh.capacity = 1;
    const double zero = 0.0;
    const int32_t izero = 0;
    sh.x = sh.y = sh.z = &zero;
    sh.typei = &izero;
    if (qphix) sh.phix.data = reps[0].phix;
    bromoc_batch *b = new bromoc_batch();
    b->device = device;
    b->sys = *s;
    b->nrep = nrep;
    b->total = total;
    StepParams sp{};
    int st = shared_context(&sh, device, &b->shared, &sp);
    if (st) {
        delete b;
        return st;
    }
    auto cleanup = [&](int code) { bromoc_batch_destroy(b); return code; };
    if (hipSetDevice(device) != hipSuccess) return cleanup(BROMOC_E_HIP);
    if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess)
        return cleanup(BROMOC_E_HIP);
#define ACHK(expr) do { if ((expr) != hipSuccess) return cleanup(BROMOC_E_HIP); } while (0)
    auto &al = b->allocs;
    b->h_off.resize(nrep);
    b->h_cap.resize(nrep);
    b->h_nfix.resize(nrep);
    b->h_nbuf.resize(nrep);
    b->h_probofs.resize(nrep);
    std::vector<int32_t> ntot(nrep);
    int64_t o = 0, po = 0;
    b->gstride = gmax + 1;
    for (int r = 0; r < nrep; r++) {
        b->h_off[r] = (int32_t)o;
        b->h_cap[r] = reps[r].capacity;
        b->h_nfix[r] = reps[r].nfix;
        b->h_nbuf[r] = reps[r].gcmc ? reps[r].gcmc->nbuffer : 0;
        b->h_probofs[r] = po;
        ntot[r] = reps[r].ntot;
        o += reps[r].capacity;
        po += (int64_t)b->h_nbuf[r] * (reps[r].capacity + 1);
    }
    std::vector<int32_t> order(nrep);
    for (int r = 0; r < nrep; r++) order[r] = r;
    std::stable_sort(order.begin(), order.end(),
                     [&](int a, int c) { return b->h_cap[a] > b->h_cap[c]; });
    // particles
    std::vector<double4> p4(total, make_double4(0.0, 0.0, 0.0, 0.0));
    std::vector<int32_t> ty(total, 0), ibuf(total, 0);
    for (int r = 0; r < nrep; r++) {
        const bromoc_replica &R = reps[r];
        for (int i = 0; i < R.ntot; i++) {
            const int64_t k = b->h_off[r] + i;
            const int t2 = s->nwtype[std::abs(R.typei[i])];
            p4[k] = make_double4(R.x[i], R.y[i], R.z[i], pack_t2(t2));
            ty[k] = R.typei[i];
            if (R.gcmc && R.ibuffer) ibuf[k] = R.ibuffer[i];
        }
    }
    for (int q = 0; q < 2; q++) ACHK(bupload(al, &b->pos[q], p4.data(), total));
    BatchParams &B = b->base;
    B.sp = sp;
    B.sp.ntargets = 0;
    for (int r = 0; r < nrep; r++) B.sp.ntargets += reps[r].capacity - reps[r].nfix;
    B.nrep = nrep;
    int32_t *d_i = nullptr;
    // the work items: every slot that can hold a moving ion, replicas by decreasing capacity
    {
        std::vector<int2> items;
        items.reserve(B.sp.ntargets);
        for (int r : order)
            for (int t = reps[r].nfix; t < reps[r].capacity; t++) items.push_back(make_int2(r, t));
        int2 *d_it = nullptr;
        ACHK(bupload(al, &d_it, items.data(), items.size()));
        B.items = d_it;
        B.nitems = (int)items.size();
        const size_t row = 3 * sizeof(double) * std::max<size_t>(items.size(), 1);
        b->noise_rows = (int)std::min<size_t>(BATCH_NOISE_ROWS, std::max<size_t>(1, BATCH_NOISE_BYTES / row));
        ACHK(balloc(al, &B.noise, b->noise_rows * 3 * std::max<size_t>(items.size(), 1)));
    }
    ACHK(bupload(al, &d_i, b->h_off.data(), nrep)); B.off = d_i;
    ACHK(bupload(al, &d_i, b->h_cap.data(), nrep)); B.cap = d_i;
    ACHK(bupload(al, &d_i, b->h_nfix.data(), nrep)); B.nfix = d_i;
    ACHK(bupload(al, &B.ntot, ntot.data(), nrep));
    ACHK(balloc(al, &B.queue, 2));
    ACHK(bupload(al, &B.typei, ty.data(), total));
    ACHK(bupload(al, &B.ibuffer, ibuf.data(), total));
    ACHK(balloc(al, &B.fx, total));
    ACHK(balloc(al, &B.fy, total));
    ACHK(balloc(al, &B.fz, total));
    ACHK(balloc(al, &B.epart, (size_t)NE * total));
    B.ecap = total;
    // static fields: one allocation per replica, a device table of their addresses
    {
        std::vector<const float *> tab(nrep, nullptr);
        if (qphix) {
            const size_t n = (size_t)s->phix.nclx * s->phix.ncly * s->phix.nclz;
            for (int r = 0; r < nrep; r++) {
                float *d = nullptr;
                ACHK(bupload(al, &d, reps[r].phix, n));
                tab[r] = d;
            }
        }
        const float **d_tab = nullptr;
        ACHK(bupload(al, (const float ***)&d_tab, (const float **)tab.data(), nrep));
        B.phix = d_tab;
    }
    const int nt = std::max(1, s->ntype - s->nold), np = std::max(1, s->cntpts);
    b->flux_stride = nt * np;
    b->warn_stride = s->nttyp + 1;
    B.flux_stride = b->flux_stride;
    B.warn_stride = b->warn_stride;
    ACHK(balloc(al, &B.nfwd, (size_t)nrep * b->flux_stride));
    ACHK(balloc(al, &B.nbwd, (size_t)nrep * b->flux_stride));
    ACHK(balloc(al, &B.warn, (size_t)nrep * b->warn_stride));
    ACHK(balloc(al, &b->warn_scratch, (size_t)nrep * b->warn_stride));
    // GCMC buffers, [nrep][gstride] with entry 0 unused as in grandmod
    {
        const int gs = b->gstride;
        std::vector<int32_t> ibf((size_t)nrep * gs, 0), tot((size_t)nrep * gs, 0), nat((size_t)nrep * gs, 0);
        std::vector<double> av((size_t)nrep * gs, 0.0), mu_((size_t)nrep * gs, 0.0),
            kb_((size_t)nrep * gs, 0.0), zl((size_t)nrep * gs, 0.0), zh((size_t)nrep * gs, 0.0);
        std::vector<int8_t> bi((size_t)nrep * gs, 0);
        std::vector<double> box((size_t)nrep * 6, 0.0);
        for (int r = 0; r < nrep; r++) {
            const bromoc_gcmc *G = reps[r].gcmc;
            if (!G) continue;
            for (int q = 1; q <= G->nbuffer; q++) {
                const size_t k = (size_t)r * gs + q;
                ibf[k] = G->ibfftyp[q]; tot[k] = G->ntotat[q]; av[k] = G->avnum[q];
                mu_[k] = G->mu[q]; kb_[k] = G->kb[q]; zl[k] = G->lzmin[q]; zh[k] = G->lzmax[q];
                bi[k] = G->bufferbias[q]; nat[k] = reps[r].nat[q];
            }
            double *bx = box.data() + 6 * (size_t)r;
            bx[0] = G->lx; bx[1] = G->ly; bx[2] = G->cx; bx[3] = G->cy; bx[4] = G->cz; bx[5] = G->ikbt;
        }
        ACHK(bupload(al, &d_i, b->h_nbuf.data(), nrep)); B.nbuf = d_i;
        ACHK(bupload(al, &d_i, ibf.data(), ibf.size())); B.ibfftyp = d_i;
        ACHK(bupload(al, &d_i, tot.data(), tot.size())); B.ntotat = d_i;
        double *d_d = nullptr;
        ACHK(bupload(al, &d_d, av.data(), av.size())); B.avnum = d_d;
        ACHK(bupload(al, &d_d, mu_.data(), mu_.size())); B.mu = d_d;
        ACHK(bupload(al, &d_d, kb_.data(), kb_.size())); B.kb = d_d;
        ACHK(bupload(al, &d_d, zl.data(), zl.size())); B.lzmin = d_d;
        ACHK(bupload(al, &d_d, zh.data(), zh.size())); B.lzmax = d_d;
        int8_t *d_b = nullptr;
        ACHK(bupload(al, &d_b, bi.data(), bi.size())); B.bias = d_b;
        ACHK(bupload(al, &d_d, box.data(), box.size())); B.gbox = d_d;
        ACHK(bupload(al, &B.nat, nat.data(), nat.size()));
        B.gstride = gs;
        ACHK(balloc(al, &B.prob, (size_t)std::max<int64_t>(po, 1)));
        int64_t *d_l = nullptr;
        ACHK(bupload(al, &d_l, b->h_probofs.data(), nrep)); B.probofs = d_l;
        ACHK(balloc(al, &B.gener, nrep));
    }
    ACHK(balloc(al, &B.ctl, 8));
    ACHK(balloc(al, &b->ered, (size_t)nrep * NE));
#undef ACHK
    *out = b;
    return BROMOC_OK;
}

int bromoc_batch_run(bromoc_batch *b, int32_t nsteps, uint64_t seed, uint64_t counter0,
                     int32_t gcmc_every, int32_t ngcmc, uint64_t cycle0,
                     bromoc_energies *energies) {
    if (!b || nsteps < 0 || gcmc_every < 0 || ngcmc < 0) return BROMOC_E_ARG;
    (void)hipSetDevice(b->device);
    int st = batch_autotune(b);
    if (st) return st;
    b->h_ctl[0] = 0; b->h_ctl[1] = (int64_t)counter0; b->h_ctl[2] = 0; b->h_ctl[3] = (int64_t)seed;
    b->h_ctl[4] = 0; b->h_ctl[5] = 0; b->h_ctl[6] = (int64_t)cycle0; b->h_ctl[7] = 0;
    BCHK(b, hipMemcpyAsync(b->base.ctl, b->h_ctl, sizeof(b->h_ctl), hipMemcpyHostToDevice, b->stream));
    const int32_t qz[2] = {0, 0};
    BCHK(b, hipMemcpyAsync(b->base.queue, qz, sizeof(qz), hipMemcpyHostToDevice, b->stream));
    const bool gc = gcmc_every > 0 && ngcmc > 0;
    // one unit: [GRAND] + len steps; whole units replay a captured graph
    const int len = gc ? gcmc_every : BATCH_GRAPH_K;
    int done = 0;
    auto unit_direct = [&](int nst, bool with_gcmc, bool last_energy) -> int {
        if (with_gcmc) {
            BatchParams p = params_now(b);
            p.ngcmc = ngcmc;
            BCHK(b, enqueue_batch_gcmc(p, b->stream));
        }
        for (int k = 0; k < nst; k++) {
            BatchParams p = params_now(b);
            p.mode = 1;
            p.noise_row = k % b->noise_rows;
            if (p.noise_row == 0)
                BCHK(b, enqueue_batch_noise(p, std::min(b->noise_rows, nst - k), b->stream));
            const bool wr = last_energy && k == nst - 1;
            p.write_energy = wr ? 1 : 0;
            p.write_forces = wr ? 1 : 0;
            BCHK(b, launch_batch_step(p, b->blocks, b->lanes, b->stream));
            b->cur ^= 1;
        }
        return BROMOC_OK;
    };
    static const bool graphs_on = [] {
        const char *e = std::getenv("BROMOC_GRAPH");
        return !(e && e[0] == '0');
    }();
    while (done < nsteps) {
        const int nst = std::min(len, nsteps - done);
        const bool last = done + nst >= nsteps;
        const bool with_gcmc = gc && (done % gcmc_every == 0);
        if (!graphs_on || nst < len || (last && energies)) {
            st = unit_direct(nst, with_gcmc, last && energies != nullptr);
            if (st) return st;
            done += nst;
            continue;
        }
        bromoc_batch::Graph &g = b->graph[b->cur];
        const int gflag = with_gcmc ? 1 : 0;
        if (!g.exec || g.len != len || g.gcmc != gflag || g.ngcmc != ngcmc ||
            g.blocks != b->blocks || g.lanes != b->lanes) {
            if (g.exec) (void)hipGraphExecDestroy(g.exec);
            g.exec = nullptr;
            const int cur0 = b->cur;
            BCHK(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
            int cst = unit_direct(len, with_gcmc, false);
            hipGraph_t graph = nullptr;
            hipError_t ce = hipStreamEndCapture(b->stream, &graph);
            b->cur = cur0;
            if (cst) return cst;
            BCHK(b, ce);
            hipError_t ie = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            BCHK(b, ie);
            g.len = len; g.gcmc = gflag; g.ngcmc = ngcmc; g.blocks = b->blocks;
            g.lanes = b->lanes;
        }
        BCHK(b, hipGraphLaunch(g.exec, b->stream));
        if (len & 1) b->cur ^= 1;
        done += nst;
    }
    st = batch_sync(b);
    if (st) return st;
    st = batch_check_flags(b);
    if (st) return st;
    if (energies) {
        BCHK(b, launch_batch_reduce(params_now(b), b->ered, b->stream));
        std::vector<double> r((size_t)b->nrep * NE);
        BCHK(b, hipMemcpyAsync(r.data(), b->ered, r.size() * sizeof(double), hipMemcpyDeviceToHost, b->stream));
        st = batch_sync(b);
        if (st) return st;
        for (int k = 0; k < b->nrep; k++) batch_energies(r.data() + (size_t)k * NE, &energies[k]);
    }
    return BROMOC_OK;
}

int bromoc_batch_energy(bromoc_batch *b, bromoc_energies *energies) {
    if (!b || !energies) return BROMOC_E_ARG;
    (void)hipSetDevice(b->device);
    int st = batch_autotune(b);
    if (st) return st;
    BatchParams p = params_now(b);
    p.mode = 0;
    p.write_energy = 1;
    p.write_forces = 1;
    BCHK(b, launch_batch_step(p, b->blocks, b->lanes, b->stream));
    BCHK(b, launch_batch_reduce(p, b->ered, b->stream));
    std::vector<double> r((size_t)b->nrep * NE);
    BCHK(b, hipMemcpyAsync(r.data(), b->ered, r.size() * sizeof(double), hipMemcpyDeviceToHost, b->stream));
    st = batch_sync(b);
    if (st) return st;
    for (int k = 0; k < b->nrep; k++) batch_energies(r.data() + (size_t)k * NE, &energies[k]);
    return BROMOC_OK;
}

int bromoc_batch_get(bromoc_batch *b, int32_t r, double *x, double *y, double *z, int32_t *typei,
                     int32_t *ntot, int32_t *ibuffer, int32_t *nat, double *gcmc_ener) {
    if (!b || r < 0 || r >= b->nrep) return BROMOC_E_ARG;
    (void)hipSetDevice(b->device);
    // everything in one launch through pinned memory, laid out by the replica's capacity; a
    // replica of more than BATCH_GET_SLOTS particles in several, so that what is pinned is bounded
    const size_t cap = std::min<size_t>(b->h_cap[r], BATCH_GET_SLOTS), nb = b->h_nbuf[r];
    const size_t bytes = sizeof(double) * (3 * cap + 1) + sizeof(int32_t) * (2 * cap + nb + 1);
    if (bytes > b->pin_cap) {
        if (b->pin) (void)hipHostFree(b->pin);
        b->pin = nullptr;
        b->pin_cap = 0;
        BCHK(b, hipHostMalloc(&b->pin, bytes));
        b->pin_cap = bytes;
    }
    StageReplica a{};
    const BatchParams &B = b->base;
    a.r = r;
    a.nbuf = (int32_t)nb;
    a.max = (int32_t)cap;
    a.ntot = B.ntot; a.off = B.off;
    a.pos = b->pos[b->cur];
    a.typei = B.typei; a.ibuffer = B.ibuffer;
    a.nat = B.nat + (size_t)r * b->gstride + 1;
    a.gener = B.gener;
    a.o_ener = (double *)b->pin;
    a.o_x = a.o_ener + 1; a.o_y = a.o_x + cap; a.o_z = a.o_y + cap;
    a.o_n = (int32_t *)(a.o_z + cap);
    a.o_nat = a.o_n + 1; a.o_ty = a.o_nat + nb; a.o_ib = a.o_ty + cap;
    int32_t n = 0;
    do {
        BCHK(b, launch_stage_replica(a, b->stream));
        int st = batch_sync(b);
        if (st) return st;
        n = a.o_n[0];
        const int32_t m = std::min(n - a.lo, a.max);
        if (x) std::copy(a.o_x, a.o_x + m, x + a.lo);
        if (y) std::copy(a.o_y, a.o_y + m, y + a.lo);
        if (z) std::copy(a.o_z, a.o_z + m, z + a.lo);
        if (typei) std::copy(a.o_ty, a.o_ty + m, typei + a.lo);
        if (ibuffer) std::copy(a.o_ib, a.o_ib + m, ibuffer + a.lo);
        a.lo += m;
    } while (a.lo < n);
    if (nat) {
        nat[0] = 0;
        std::copy(a.o_nat, a.o_nat + nb, nat + 1);
    }
    if (gcmc_ener) *gcmc_ener = a.o_ener[0];
    if (ntot) *ntot = n;
    return BROMOC_OK;
}

int bromoc_batch_get_forces(bromoc_batch *b, int32_t r, double *fx, double *fy, double *fz) {
    if (!b || r < 0 || r >= b->nrep || !fx || !fy || !fz) return BROMOC_E_ARG;
    (void)hipSetDevice(b->device);
    int32_t n = 0;
    BCHK(b, hipMemcpy(&n, b->base.ntot + r, sizeof(n), hipMemcpyDeviceToHost));
    const int64_t off = b->h_off[r];
    if (n) {
        BCHK(b, hipMemcpy(fx, b->base.fx + off, sizeof(double) * n, hipMemcpyDeviceToHost));
        BCHK(b, hipMemcpy(fy, b->base.fy + off, sizeof(double) * n, hipMemcpyDeviceToHost));
        BCHK(b, hipMemcpy(fz, b->base.fz + off, sizeof(double) * n, hipMemcpyDeviceToHost));
    }
    return BROMOC_OK;
}

int bromoc_batch_get_flux(bromoc_batch *b, int32_t r, int32_t *nforward, int32_t *nbackward) {
    if (!b || r < 0 || r >= b->nrep || !nforward || !nbackward) return BROMOC_E_ARG;
    (void)hipSetDevice(b->device);
    const int nt = b->sys.ntype - b->sys.nold, np = b->sys.cntpts;
    if (nt <= 0 || np <= 0) return BROMOC_OK;
    const size_t o = (size_t)r * b->flux_stride;
    BCHK(b, hipMemcpy(nforward, b->base.nfwd + o, sizeof(int32_t) * nt * np, hipMemcpyDeviceToHost));
    BCHK(b, hipMemcpy(nbackward, b->base.nbwd + o, sizeof(int32_t) * nt * np, hipMemcpyDeviceToHost));
    return BROMOC_OK;
}

int bromoc_batch_get_prob(bromoc_batch *b, int32_t r, int32_t *prob) {
    if (!b || r < 0 || r >= b->nrep || !prob) return BROMOC_E_ARG;
    (void)hipSetDevice(b->device);
    const size_t n = (size_t)b->h_nbuf[r] * (b->h_cap[r] + 1);
    if (n) BCHK(b, hipMemcpy(prob, b->base.prob + b->h_probofs[r], sizeof(int32_t) * n, hipMemcpyDeviceToHost));
    return BROMOC_OK;
}

int bromoc_batch_time_steps(bromoc_batch *b, int32_t nsteps, uint64_t seed, uint64_t counter0,
                            double *total_ms, double *kernel_ms) {
    if (!b || nsteps <= 0 || !total_ms || !kernel_ms) return BROMOC_E_ARG;
    (void)hipSetDevice(b->device);
    int st = batch_autotune(b);
    if (st) return st;
    b->h_ctl[0] = 0; b->h_ctl[1] = (int64_t)counter0; b->h_ctl[3] = (int64_t)seed;
    BCHK(b, hipMemcpyAsync(b->base.ctl, b->h_ctl, sizeof(b->h_ctl), hipMemcpyHostToDevice, b->stream));
    std::vector<hipEvent_t> ev(2 * nsteps);
    for (auto &e : ev) BCHK(b, hipEventCreate(&e));
    for (int k = 0; k < nsteps; k++) {
        BatchParams p = params_now(b);
        p.mode = 1;
        p.noise_row = 0;
        BCHK(b, enqueue_batch_noise(p, 1, b->stream));
        BCHK(b, hipEventRecord(ev[2 * k], b->stream));
        BCHK(b, launch_batch_step(p, b->blocks, b->lanes, b->stream));
        BCHK(b, hipEventRecord(ev[2 * k + 1], b->stream));
        b->cur ^= 1;
    }
    st = batch_sync(b);
    if (st) return st;
    double sum = 0.0;
    for (int k = 0; k < nsteps; k++) {
        float ms = 0.f;
        BCHK(b, hipEventElapsedTime(&ms, ev[2 * k], ev[2 * k + 1]));
        sum += ms;
    }
    float all = 0.f;
    BCHK(b, hipEventElapsedTime(&all, ev[0], ev[2 * nsteps - 1]));
    for (auto &e : ev) (void)hipEventDestroy(e);
    *total_ms = all;
    *kernel_ms = sum / nsteps;
    return BROMOC_OK;
}

int bromoc_batch_get_tuning(bromoc_batch *b, int32_t *blocks, int32_t *lanes) {
    if (!b || !blocks || !lanes) return BROMOC_E_ARG;
    (void)hipSetDevice(b->device);
    int st = batch_autotune(b);
    if (st) return st;
    *blocks = b->blocks;
    *lanes = b->lanes;
    return BROMOC_OK;
}

}  // extern "C"
