// tiles.hip -- tile mode of the BD step: every unordered particle pair evaluated once.
//
// The reference's ENERGY visits each ion-ion pair once (energy.mono.f90:117-194) and
// applies Newton's third law; its reaction-field cross term does the same for each ion
// pair (rfpar.f90:177-223), and the ion-DNA loop each site-ion pair (:584-687).  k_step
// gathers instead, every target over all partners, which costs every pair twice.  Tile
// mode keeps the reference's once-per-pair work and stays deterministic:
//
//  * the particles in tile order (sort.hip: fixed ions, sites, moving ions, each by atnam2 type,
//    each type in spatial order) are cut into tiles of TT = 64 * TPL slots; each class and type
//    begins a new tile, so a tile holds fixed ions, sites or moving ions of one type, and empty
//    slots at the end of a run;
//  * k_tiles: one wavefront per item (I, g): tile I's particles are its targets, TPL per
//    lane in registers, and the tiles J >= I of column group g (R consecutive tiles) pass by
//    in chunks of 64 partners.  A chunk's positions are staged in LDS, twice in a row, so
//    that at step k lane l reads partner l + k without wrapping; every lane takes another
//    partner, evaluates it against its TPL targets and adds the targets' shares in
//    registers.  The partners' shares travel: each lane holds the sums of the partner it is
//    evaluating and hands them to its lower neighbour after the step (DPP wavefront
//    rotation), so after 64 steps lane l holds partner l's sums -- no LDS accumulators, whose
//    read-modify-write took as long as the arithmetic.  Each pair's reaction-field cross
//    term (when the system has one) is evaluated in the same sweep;
//  * the targets' sums are written once per item, a chunk's partner sums once per (I, J): a
//    tile's rows of tpart, one per lower tile and one per group of higher ones, each written
//    once per step; pair energies go to tener[cat][item];
//  * the sweep a chunk takes depends on what it and the target tile hold.  Against a chunk
//    of moving ions there is one pair type, its parameters in scalar registers.  When no
//    partner of the chunk is within table range of the targets' bounding box (97 % of the
//    chunks at 56,000 particles) the sweep is straight-line code: the analytic tail alone,
//    no comparison, no table.  In near chunks the
//    sweep leaves the pairs in range out and notes them, a bit per pair for the target and one
//    that travels with the partner; then each lane works off its targets' bits and its
//    partner's, so the table's root, index and gather (three times the tail's arithmetic and a
//    memory round trip) are paid per pair in range and not per step that has one.  Masks
//    (the diagonal, empty slots) are a variant of their own.  The reaction-field term, when
//    every ion of both sides is either inside the grid with a nonzero srfe or outside it
//    with none, reduces to per-ion weights folded into the charges (or vanishes, when one
//    side has no ion inside); sites against moving ions have none.  Chunks with an ion inside
//    the grid where srfe is zero, whose pairs count by their order (rfpar.f90:177), take the same
//    sweeps for the pair forces and a masked one for the reaction field alone: with 5 % of the
//    cells zero, 20,000 ions 1030 -> 470 us a step (820 with both in one masked sweep, whose
//    table branch is taken at most steps).  Fixed ions against moving ones take the straight
//    sweeps unless there is a reaction field (a third of 20,000 ions fixed: 370 -> 285 us);
//    with one, and against sites, the general masked sweep;
//  * k_tfin: eight lanes per slot sum the slot's partial rows in a fixed order,
//    gather the grid corners and finish the particle as k_step does (CG-DNA list forces,
//    reaction-field gradients and self term, MEMBRANE, energies, BD update).
#include <algorithm>
#include <type_traits>

#include "device.h"

namespace bromoc {

constexpr int F_RFT = 64;   // reaction-field cross term fused into the pair sweep
// slot flags (bits above the atnam2 type, which takes the low 16): a particle (VALID), a
// site, a fixed ion, receiving pair forces (RECV), moving and inside the reaction-field grid
// (HI), a moving ion (ION); for the reaction field, a moving ion with HI and srfe != 0
// (RFON) and one with exactly one of the two (RFODD)
constexpr int SL_VALID = 1, SL_SITE = 2, SL_FIXED = 4, SL_RECV = 8, SL_HI = 16, SL_ION = 32,
              SL_RFON = 64, SL_RFODD = 128;

// Column groups of n tiles: R tiles per group, so that an item's targets (their sums, and
// the row they write) serve R tiles.  The largest R that still gives the chip several
// rounds of wavefronts, since the items' lengths differ.
int tile_run(int n) {
    for (int r = 8; r > 1; r >>= 1) {
        const int64_t g = (n + r - 1) / r;
        if (r * g * (g + 1) / 2 >= TILE_MIN_ITEMS) return r;
    }
    return 1;
}
int tile_items(int n) {
    const int r = tile_run(n), g = (n + r - 1) / r;
    return r * (g * (g + 1) / 2);
}

int tile_count(int n, int ttpl, int runs) {
    const int tt = 64 * ttpl;
    return (int)((n + (int64_t)runs * (tt - 1)) / tt);
}
size_t tile_part_doubles(int cap, int ttpl, int runs, int rf) {
    const size_t tt = 64 * (size_t)ttpl, nc = tile_count(cap, ttpl, runs);
    size_t rows = 0;   // the run length, and so the rows, follow the tiles now in use
    for (size_t n = 1; n <= nc; n++) rows = std::max(rows, (size_t)tile_row(n, n, tile_run((int)n)));
    return rows * (rf ? 5 : 3) * tt;
}
size_t tile_ener_doubles(int cap, int ttpl, int runs) {
    const size_t nc = tile_count(cap, ttpl, runs);
    size_t m = 0;
    for (size_t n = 1; n <= nc; n++)   // energies, then the tflag words
        m = std::max(m, 2 * (size_t)NTE * tile_items((int)n) +
                            ((size_t)tile_row(n, n, tile_run((int)n)) * ttpl + 1) / 2);
    return m;
}

// The particle in slot s of the tile order: position, and a word of atnam2 type and
// flags (the pair kernels' masks); with the reaction field, srfe, reff and the charge.
struct SlotInfo {
    double x, y, z, sr, rr, q;
    int tf, idx;
};

template <int FEAT>
__device__ __forceinline__ SlotInfo slot_info(const StepParams &P, int s) {
    SlotInfo o;
    const double4 pa = P.spos[s];   // an empty slot: index -1, at the box's centre
    const bool ok = __double2hiint(pa.w) >= 0;
    const int idx = ok ? __double2hiint(pa.w) : 0, t2 = __double2loint(pa.w);
    const bool site = ok && idx < P.nsites, fixed = ok && !site && idx < P.nsites + P.nfix;
    bool recv = ok && !site && !fixed;
    if constexpr ((FEAT & F_DNA) != 0) {
        if (site) recv = P.stfree[idx] != 0;
    }
    const bool ion = ok && !site && !fixed;
    int fl = (ok ? SL_VALID : 0) | (site ? SL_SITE : 0) | (fixed ? SL_FIXED : 0) |
             (recv ? SL_RECV : 0) | (ion ? SL_ION : 0);
    o.x = pa.x; o.y = pa.y; o.z = pa.z;
    o.sr = 0.0; o.rr = 0.0; o.q = 0.0;
    if constexpr ((FEAT & F_RFT) != 0) {
        if (ok && !site) {
            // (srfe, reff, inside the grid box, moving) from k_rfpar; charge in rfq.w
            const double4 ra = P.rfa[idx];
            o.sr = ra.x; o.rr = ra.y;
            o.q = P.rfq[idx].w;
            const bool hi = ra.z != 0.0 && ra.w != 0.0;
            if (hi) fl |= SL_HI;
            if (ion && hi && ra.x != 0.0) fl |= SL_RFON;
            if (ion && hi != (ra.x != 0.0)) fl |= SL_RFODD;
        }
    }
    o.tf = t2 | (fl << 16);
    o.idx = idx;
    return o;
}

// the low 8 bits of v AND-ed (OR-ed) over the wavefront
__device__ __forceinline__ int wave_and8(int v) {
    int r = 0;
#pragma unroll
    for (int b = 0; b < 8; b++)
        if (__ballot(((v >> b) & 1) == 0) == 0ull) r |= 1 << b;
    return r;
}
__device__ __forceinline__ int wave_or8(int v) {
    int r = 0;
#pragma unroll
    for (int b = 0; b < 8; b++)
        if (__ballot((v >> b) & 1) != 0ull) r |= 1 << b;
    return r;
}

// item -> (row I, group g): group g holds the rows 0 .. (g + 1) R - 1, groups in order
__device__ __forceinline__ void item_tiles(int item, int R, int &I, int &g) {
    const int h = item / R;   // g (g + 1) / 2 <= h
    int k = (int)((sqrt(8.0 * (double)h + 1.0) - 1.0) * 0.5);
    while (k > 0 && k * (k + 1) / 2 > h) k--;
    while ((k + 1) * (k + 2) / 2 <= h) k++;
    g = k;
    I = item - R * (k * (k + 1) / 2);
}

// a chunk of 64 partners staged by the wavefront, each entry twice (at p and p + 64)
template <bool RF, int TT>
struct Chunk {
    double x[2 * WAVE], y[2 * WAVE], z[2 * WAVE];
    double tx[TT], ty[TT], tz[TT];   // the targets, for the partners' pairs in range
    union {
        struct { double rr[RF ? 2 * WAVE : 1], qs[RF ? 2 * WAVE : 1]; };   // reff; weight * charge * srfe
        struct {   // the general sweep's: srfe, reff, charge, index
            double sr[RF ? 2 * WAVE : 1], rg[RF ? 2 * WAVE : 1], q[RF ? 2 * WAVE : 1];
            int ix[RF ? 2 * WAVE : 1];
        };
    };
    int tf[2 * WAVE];   // type and flags
};

// wavefronts per SIMD the registers are held to
constexpr int tile_occ(int feat, int tpl) {
    return tpl == 4 ? 2 : (feat & F_TAB) == 0 ? 2 : tpl == 1 ? ((feat & F_RFT) ? 4 : 5) : (feat & F_RFT) ? 3 : 4;
}

// k_tiles: see the file comment.  One wavefront per block: its item ends on its own.  Bound by
// FP64 issue where the system is large: 27 issue slots a far pair (four of them the reciprocal
// root's), 24 more with the reaction field, and the rotation's ten moves a step.  Measured, one
// launch (before, with LDS accumulators, per-pair table parameters and a branch per pair;
// after): 56,000 particles with the reaction field on every ion pair 3.34 -> 2.56 ms, 12,457
// particles 237 -> 177 us, 6,001 particles 55 -> 47 us.
template <int FEAT, int TPL, bool EN>
__global__ __launch_bounds__(WAVE)
__attribute__((amdgpu_waves_per_eu(tile_occ(FEAT, TPL))))
void k_tiles(StepParams P) {
    constexpr int TT = WAVE * TPL;
    constexpr bool RF = (FEAT & F_RFT) != 0, TAB = (FEAT & F_TAB) != 0;
    __shared__ Chunk<RF, TT> C;

    const int lane = threadIdx.x, item = blockIdx.x;
    const int n = P.ntile, nt1 = P.nttyp + 1, R = P.trun;
    int I, g;
    item_tiles(item, R, I, g);
    double *const eout = P.tener + 2 * (size_t)item;   // the item's pair of category 0
    auto ener_zero = [&](int cat) { eout[2 * (size_t)cat * P.titems] = eout[2 * (size_t)cat * P.titems + 1] = 0.0; };
    if (I >= n) {   // past the last tile of a partial last group
        if (EN && lane < NTE) ener_zero(lane);
        return;
    }
    // Pair energies, carried with their rounding errors: table, Coulomb, LJ, SRPMF and the
    // reaction field.  A tile holds one class, so a chunk's pairs all are of sites and ions
    // (mx) or none is, and along an item's chunks that changes at most once: targets that are
    // fixed ions, whose partners go from sites to ions.  ener_end files the first four under
    // the class that ends.  (A sum for each of the nine categories, without its error, spilled up
    // to 193 registers and lost up to two digits of the total: 392 us an ENERGY of 12,457
    // particles with the reaction field, 294 now.)
    Sum2 e0 = {0.0, 0.0}, e1 = e0, e2 = e0, e3 = e0, erf = e0;
    int eclass = -1, edone = 0;   // class of the chunks now summed; classes filed
    auto ener_out = [&](int cat, const Sum2 &v) {
        Sum2 t = {0.0, 0.0};
        if (__ballot(v.s != 0.0 || v.c != 0.0) != 0ull) t = group_sum2<WAVE>(v);
        if (lane == 0) {
            double *const d = eout + 2 * (size_t)cat * P.titems;
            d[0] = t.s;
            d[1] = isfinite(t.s) ? t.c : 0.0;   // the error of an infinite sum is not a number
        }
    };
    auto ener_end = [&](int mx) {
        ener_out(mx ? TE_EFPOTMX : TE_EFPOT, e0);
        ener_out(mx ? TE_QQMX : TE_ELEC, e1);
        ener_out(mx ? TE_VDWMX : TE_VDW, e2);
        ener_out(mx ? TE_SRPMFMX : TE_SRPMF, e3);
        e0 = e1 = e2 = e3 = Sum2{0.0, 0.0};
        edone |= 1 << mx;
    };
    const int NC = RF ? 5 : 3;
    const int J0 = max(I, g * R), J1 = min((g + 1) * R, n);
    // targets: tile I in registers
    double tx[TPL], ty[TPL], tz[TPL], tsr[TPL], trr[TPL], tq[TPL];
    int ttf[TPL], tix[TPL];
    double ax_[TPL], ay_[TPL], az_[TPL], aa_[TPL], ab_[TPL];   // aa_, ab_: general sweep
    double wa[TPL], wb[TPL], tqs[TPL];   // the weighted sweeps' A and B over their factors
    int andI = ~0, orI = 0;
#pragma unroll
    for (int u = 0; u < TPL; u++) {
        const SlotInfo o = slot_info<FEAT>(P, I * TT + lane + WAVE * u);
        tx[u] = o.x; ty[u] = o.y; tz[u] = o.z; ttf[u] = o.tf; tix[u] = o.idx;
        tsr[u] = o.sr; trr[u] = o.rr; tq[u] = o.q;
        ax_[u] = ay_[u] = az_[u] = aa_[u] = ab_[u] = wa[u] = wb[u] = 0.0;
        C.tx[lane + WAVE * u] = o.x; C.ty[lane + WAVE * u] = o.y; C.tz[lane + WAVE * u] = o.z;
        const int f = o.tf >> 16;
        tqs[u] = (f & SL_RFON) ? P.celec * o.q * o.sr : 0.0;
        andI &= (f & SL_VALID) ? f : ~SL_VALID;
        orI |= f;
    }
    const int t2I = __builtin_amdgcn_readfirstlane(ttf[0] & 0xFFFF);   // a run begins with a particle
    andI = wave_and8(andI); orI = wave_or8(orI);
    // the tile's class (every particle's: an empty slot has no say)
    const bool ionI = (orI & SL_ION) && (andI & SL_ION), siteI = (orI & SL_SITE) && (andI & SL_SITE);
    // the targets' bounding box
    double bx0 = tx[0], bx1 = tx[0], by0 = ty[0], by1 = ty[0], bz0 = tz[0], bz1 = tz[0];
#pragma unroll
    for (int u = 1; u < TPL; u++) {
        bx0 = fmin(bx0, tx[u]); bx1 = fmax(bx1, tx[u]);
        by0 = fmin(by0, ty[u]); by1 = fmax(by1, ty[u]);
        bz0 = fmin(bz0, tz[u]); bz1 = fmax(bz1, tz[u]);
    }
    bx0 = wave_min(bx0); bx1 = wave_max(bx1);
    by0 = wave_min(by0); by1 = wave_max(by1);
    bz0 = wave_min(bz0); bz1 = wave_max(bz1);
    bool rfany = false;   // the targets' reaction-field sums (A, B) may be nonzero

    for (int J = J0; J < J1; J++) {
        const bool diag = I == J;
        double *const prow = P.tpart + ((size_t)(tile_row(J, n, R) + I) * NC) * TT;
        int32_t *const pflag = P.tflag + (size_t)(tile_row(J, n, R) + I) * TPL;
#pragma unroll 1
        for (int q = 0; q < TPL; q++) {
            const SlotInfo o = slot_info<FEAT>(P, J * TT + WAVE * q + lane);
            const int pf = o.tf >> 16;
            const int andJ = wave_and8((pf & SL_VALID) ? pf : ~SL_VALID), orJ = wave_or8(pf);
            const bool ionJ = (orJ & SL_ION) && (andJ & SL_ION);
            // the sums of the partner this lane holds
            double gx = 0.0, gy = 0.0, gz = 0.0, ga = 0.0, gb = 0.0;
            bool rfsums = false;   // the chunk's A and B may be nonzero
            // sites among themselves and fixed ions among themselves have no pair
            if ((orI & SL_VALID) && (orJ & SL_VALID) && !(orI & orJ & (SL_SITE | SL_FIXED))) {
                if constexpr (EN) {
                    const int mx = ((orI | orJ) & SL_SITE) ? 1 : 0;
                    if (eclass >= 0 && eclass != mx) ener_end(eclass);
                    eclass = mx;
                }
                __builtin_amdgcn_wave_barrier();
                C.x[lane] = o.x; C.y[lane] = o.y; C.z[lane] = o.z;
                C.x[lane + WAVE] = o.x; C.y[lane + WAVE] = o.y; C.z[lane + WAVE] = o.z;
                // the straight sweeps for the pair forces (k_tfin has no use for the sums of a fixed ion
                // without a reaction field), the reaction field by weights, or by a sweep of its own
                // the pair type: a run's slots are filled from its start
                const int t2J = __builtin_amdgcn_readfirstlane(o.tf & 0xFFFF);
                const DevPair &pr = P.rows[t2I * nt1 + t2J];
                const bool fast = ionJ && (siteI || ionI || !RF);
                const bool rfodd = RF && ionI && ionJ && ((orI | orJ) & SL_RFODD) && ((orI | orJ) & SL_RFON);
                const bool rfw = RF && ionI && !rfodd && (orI & SL_RFON) && (orJ & SL_RFON);
                if (fast) {
                    const bool mask = diag || !(andI & SL_VALID) || !(andJ & SL_VALID);
                    const uint64_t pval = __ballot(pf & SL_VALID);
                    const double s3 = wave_uniform(pr.sc3), s6 = wave_uniform(6.0 * pr.sc3);
                    const double fc = wave_uniform(pr.fct), hi = wave_uniform(pr.dm2hi);
                    const int fl = __builtin_amdgcn_readfirstlane(pr.flags);
                    // a partner within table range of the targets' box?
                    const double ex = fmax(fmax(bx0 - o.x, o.x - bx1), 0.0);
                    const double ey = fmax(fmax(by0 - o.y, o.y - by1), 0.0);
                    const double ez = fmax(fmax(bz0 - o.z, o.z - bz1), 0.0);
                    const bool far = __ballot(!(ex * ex + ey * ey + ez * ez > hi * (1.0 + 1e-9))) == 0ull;
                    if constexpr (RF) {
                        if (rfw) {
                            const double w = (pf & SL_RFON) ? o.q * o.sr : 0.0;
                            C.rr[lane] = o.rr; C.qs[lane] = w;
                            C.rr[lane + WAVE] = o.rr; C.qs[lane + WAVE] = w;
                        }
                    }
                    // LDS operations of one wavefront complete in order; the fences keep the
                    // compiler from moving them across
                    __atomic_signal_fence(__ATOMIC_SEQ_CST);
                    __builtin_amdgcn_wave_barrier();
                    double es = 0.0, er = 0.0;   // energies of a step's TPL pairs, added at its end
                    auto step_energies = [&] {
                        sum2_fast(e0, es);
                        if constexpr (RF) sum2_fast(erf, er);
                        es = er = 0.0;
                    };
                    // The reaction-field term of a pair (rfpar.f90:177-223) with R = reff reff',
                    // w = 1/sqrt(R^2 + d2), Q = celec q srfe q' srfe' (ions' weights in qs):
                    // energy Q R w; force factor Q w^3 R; A of a target sums R w (q' srfe') and
                    // takes its factor celec q at the end, B sums Q w^3 (d2 + R / 2) reff'.
                    auto rf_pair = [&](auto masked, int u, double d2, double prr, double pqs, double &f) {
                        const double rp = trr[u] * prr, s2 = fma(rp, rp, d2);
                        const double w = decltype(masked)::value ? rsqrt_s26(s2) : rsqrt_c3(s2);
                        const double a = rp * w, Q = tqs[u] * pqs;
                        const double a2 = Q * w * (w * w);
                        const double a3 = a2 * fma(rp, 0.5, d2);
                        if constexpr (EN) er = fma(Q, a, er);
                        wa[u] = fma(a, pqs, wa[u]);
                        wb[u] = fma(a3, prr, wb[u]);
                        ga = fma(a, tqs[u], ga);
                        gb = fma(a3, trr[u], gb);
                        f = fma(a2, rp, f);
                    };
                    auto add = [&](int u, double f, double dx, double dy, double dz) {
                        ax_[u] = fma(f, dx, ax_[u]);
                        ay_[u] = fma(f, dy, ay_[u]);
                        az_[u] = fma(f, dz, az_[u]);
                        gx = fma(-f, dx, gx);
                        gy = fma(-f, dy, gy);
                        gz = fma(-f, dz, gz);
                    };
                    // no pair in range: the tail alone
                    auto sweep_far = [&](auto rf_on) {
                        constexpr bool RFW = decltype(rf_on)::value;
#pragma unroll (TPL == 1 ? 4 : TPL == 2 ? 2 : 1)
                        for (int k = 0; k < WAVE; k++) {
                            const double px = C.x[lane + k], py = C.y[lane + k], pz = C.z[lane + k];
                            double prr = 0.0, pqs = 0.0;
                            if constexpr (RFW) { prr = C.rr[lane + k]; pqs = C.qs[lane + k]; }
#pragma unroll
                            for (int u = 0; u < TPL; u++) {
                                const double dx = tx[u] - px, dy = ty[u] - py, dz = tz[u] - pz;
                                const double d2 = pair_d2(dx, dy, dz);
                                const double r = rsqrt_c3(d2), i2 = r * r, i4 = i2 * i2, fr = fc * r;
                                double f = fma(s6 * i2, i4, fr) * i2;
                                if constexpr (EN) es += fma(s3 * i2, i4, fr);
                                if constexpr (RFW) rf_pair(std::false_type{}, u, d2, prr, pqs, f);
                                add(u, f, dx, dy, dz);
                            }
                            if constexpr (EN) step_energies();
                            gx = wave_next(gx); gy = wave_next(gy); gz = wave_next(gz);
                            if constexpr (RFW) { ga = wave_next(ga); gb = wave_next(gb); }
                        }
                    };
                    // a step's mask: a pair counts when both slots hold a particle and, on the
                    // diagonal, once: against its own chunk a lane takes the first half of the
                    // rotation, against higher chunks all of it, against lower ones none
                    auto counts = [&](int u, int k) {
                        const bool pv = (pval >> ((lane + k) & (WAVE - 1))) & 1ull;
                        bool c = pv && ((ttf[u] >> 16) & SL_VALID);
                        if (diag) c = c && (u < q || (u == q && k > 0 && (k < 32 || (k == 32 && lane < 32))));
                        return c;
                    };
                    const int kend = diag && q == 0 ? 33 : WAVE;
                    // some pair may be in range: the tail of the others, and the bits (k: the
                    // pair met at step k) of those, per target and per partner
                    auto sweep_near = [&](auto rf_on, auto mask_on) {
                        constexpr bool RFW = decltype(rf_on)::value;
                        constexpr bool MASK = decltype(mask_on)::value;
                        uint32_t tm[2][TPL], pm[2][TPL];
#pragma unroll
                        for (int w = 0; w < 2; w++) {
#pragma unroll
                            for (int u = 0; u < TPL; u++) tm[w][u] = pm[w][u] = 0u;
                            const int k1 = MASK ? min(kend, 32 * (w + 1)) : 32 * (w + 1);
#pragma unroll 1
                            for (int k = 32 * w; k < k1; k++) {
                                const double px = C.x[lane + k], py = C.y[lane + k], pz = C.z[lane + k];
                                const uint32_t bit = 1u << (k & 31);
                                double prr = 0.0, pqs = 0.0;
                                if constexpr (RFW) { prr = C.rr[lane + k]; pqs = C.qs[lane + k]; }
#pragma unroll
                                for (int u = 0; u < TPL; u++) {
                                    const double dx = tx[u] - px, dy = ty[u] - py, dz = tz[u] - pz;
                                    double d2 = pair_d2(dx, dy, dz);
                                    const bool on = !MASK || counts(u, k);
                                    if constexpr (MASK) d2 = on ? d2 : 1.0;
                                    const bool near = on && d2 <= hi;
                                    const double r = MASK ? rsqrt_s26(d2) : rsqrt_c3(d2), i2 = r * r, i4 = i2 * i2, fr = fc * r;
                                    double f = fma(s6 * i2, i4, fr) * i2;
                                    f = on && !near ? f : 0.0;
                                    if constexpr (EN) es += on && !near ? fma(s3 * i2, i4, fr) : 0.0;
                                    const uint32_t nb = near ? bit : 0u;
                                    tm[w][u] |= nb;
                                    pm[w][u] |= nb;
                                    // a masked pair: zero weight and reff, so every term is zero
                                    if constexpr (RFW) rf_pair(mask_on, u, d2, on ? prr : 0.0, on ? pqs : 0.0, f);
                                    add(u, f, dx, dy, dz);
                                    pm[w][u] = wave_next(pm[w][u]);
                                }
                                if constexpr (EN) step_energies();
                                gx = wave_next(gx); gy = wave_next(gy); gz = wave_next(gz);
                                if constexpr (RFW) { ga = wave_next(ga); gb = wave_next(gb); }
                            }
                            if constexpr (MASK) {   // the steps left out of a half rotation
#pragma unroll 1
                                for (int k = max(k1, 32 * w); k < 32 * (w + 1); k++) {
                                    gx = wave_next(gx); gy = wave_next(gy); gz = wave_next(gz);
                                    if constexpr (RFW) { ga = wave_next(ga); gb = wave_next(gb); }
#pragma unroll
                                    for (int u = 0; u < TPL; u++) pm[w][u] = wave_next(pm[w][u]);
                                }
                            }
                        }
                        // after its 32 steps the second word is home (lane l holds partner
                        // l's), the first half way round
#pragma unroll
                        for (int u = 0; u < TPL; u++)
                            pm[0][u] = __shfl(pm[0][u], (lane + 32) & (WAVE - 1), WAVE);
                        const double lo = wave_uniform(pr.dm2lo), dmi = wave_uniform(pr.dmi);
                        const int nxi = __builtin_amdgcn_readfirstlane(pr.nxi);
                        const int nlast = __builtin_amdgcn_readfirstlane(pr.nlast);
                        // the lane's pairs in range with the entries (lane + sgn k) of the
                        // staged positions sx, sy, sz, two at a time; energy when it is the target
                        auto work_off = [&](uint64_t m, int sgn, double x0, double y0, double z0,
                                            const double *sx, const double *sy, const double *sz,
                                            double &fx, double &fy, double &fz, bool head) {
                            while (m) {
                                double dx[2], dy[2], dz[2], d2[2], ri[2], k0[2], k1[2], k2[2];
                                const bool two = (m & (m - 1)) != 0ull;
#pragma unroll
                                for (int h = 0; h < 2; h++) {
                                    const int k = __ffsll((unsigned long long)m) - 1;
                                    if (h == 0 && two) m &= m - 1;
                                    const int p = (lane + sgn * k) & (WAVE - 1);
                                    dx[h] = x0 - sx[p]; dy[h] = y0 - sy[p]; dz[h] = z0 - sz[p];
                                    d2[h] = pair_d2(dx[h], dy[h], dz[h]);
                                    ri[h] = rsqrt_s26(d2[h]);
                                    int kn = (int)((root_of(d2[h], ri[h]) - dmi) * P.ires) + nxi;
                                    kn = min(max(kn, nxi), nlast);
                                    const double *kp = reinterpret_cast<const double *>(P.ep + kn);
                                    if constexpr (EN) k0[h] = kp[0];
                                    k1[h] = kp[1];
                                    k2[h] = kp[2];
                                }
                                m &= m - 1;
#pragma unroll
                                for (int h = 0; h < 2; h++) {
                                    double f = -k1[h] * ri[h] - 2.0 * k2[h], y = 0.0;
                                    if constexpr (EN) {
                                        const double x = root_of(d2[h], ri[h]);
                                        y = k0[h] + x * (k1[h] + x * k2[h]);
                                    }
                                    if (d2[h] < lo) f = pair_wall(pr, ri[h], y);
                                    if (h == 1 && !two) f = y = 0.0;
                                    fx = fma(f, dx[h], fx); fy = fma(f, dy[h], fy); fz = fma(f, dz[h], fz);
                                    if constexpr (EN) { if (head) sum2_add(e0, y); }
                                }
                            }
                        };
#pragma unroll
                        for (int u = 0; u < TPL; u++) {
                            const uint64_t mt = tm[0][u] | ((uint64_t)tm[1][u] << 32);
                            const uint64_t mp = pm[0][u] | ((uint64_t)pm[1][u] << 32);
                            work_off(mt, 1, tx[u], ty[u], tz[u], C.x, C.y, C.z, ax_[u], ay_[u], az_[u], true);
                            work_off(mp, -1, o.x, o.y, o.z, C.tx + WAVE * u, C.ty + WAVE * u, C.tz + WAVE * u,
                                     gx, gy, gz, false);
                        }
                    };
                    // analytic pairs
                    auto sweep_analytic = [&](auto rf_on) {
                        constexpr bool RFW = decltype(rf_on)::value;
#pragma unroll 1
                        for (int k = 0; k < WAVE; k++) {
                            const double px = C.x[lane + k], py = C.y[lane + k], pz = C.z[lane + k];
                            double prr = 0.0, pqs = 0.0;
                            if constexpr (RFW) { prr = C.rr[lane + k]; pqs = C.qs[lane + k]; }
#pragma unroll
                            for (int u = 0; u < TPL; u++) {
                                const double dx = tx[u] - px, dy = ty[u] - py, dz = tz[u] - pz;
                                const bool on = !mask || counts(u, k);
                                const double d2 = on ? pair_d2(dx, dy, dz) : 1.0;
                                double q0 = 0.0, q1 = 0.0, q2 = 0.0;
                                double f = pair_analytic(pr, P, d2, q0, q1, q2);
                                f = on ? f : 0.0;
                                if constexpr (EN) {
                                    sum2_fast(e1, on ? q0 : 0.0);
                                    sum2_fast(e2, on ? q1 : 0.0);
                                    sum2_fast(e3, on ? q2 : 0.0);
                                }
                                if constexpr (RFW) rf_pair(std::true_type{}, u, d2, on ? prr : 0.0, on ? pqs : 0.0, f);
                                add(u, f, dx, dy, dz);
                            }
                            if constexpr (EN && RFW) { sum2_fast(erf, er); er = 0.0; }
                            gx = wave_next(gx); gy = wave_next(gy); gz = wave_next(gz);
                            if constexpr (RFW) { ga = wave_next(ga); gb = wave_next(gb); }
                        }
                    };
                    auto pick = [&](auto rf_on) {
                        if constexpr (!TAB) {
                            if (!(fl & PF_EFPOT)) { sweep_analytic(rf_on); return; }
                        }
                        if (mask) sweep_near(rf_on, std::true_type{});
                        else if (!far) sweep_near(rf_on, std::false_type{});
                        else sweep_far(rf_on);
                    };
                    if (RF && rfw) {
                        rfsums = true;
                        pick(std::bool_constant<RF>{});
                        // the partners' own factors
                        ga *= (pf & SL_RFON) ? -o.q : 0.0;
                        gb = -gb;
                    } else {
                        pick(std::false_type{});
                    }
                }
                if (!fast || rfodd) {
                    // the reads above before this staging (the weights share its memory)
                    __atomic_signal_fence(__ATOMIC_SEQ_CST);
                    __builtin_amdgcn_wave_barrier();
                    C.tf[lane] = o.tf; C.tf[lane + WAVE] = o.tf;
                    if constexpr (RF) {
                        C.sr[lane] = o.sr; C.rg[lane] = o.rr; C.q[lane] = o.q; C.ix[lane] = o.idx;
                        C.sr[lane + WAVE] = o.sr; C.rg[lane + WAVE] = o.rr; C.q[lane + WAVE] = o.q;
                        C.ix[lane + WAVE] = o.idx;
                    }
                    __atomic_signal_fence(__ATOMIC_SEQ_CST);
                    __builtin_amdgcn_wave_barrier();
                    rfsums = RF;
                    auto general = [&](auto pairs_on) {
                        constexpr bool PAIRS = decltype(pairs_on)::value;
#pragma unroll 1
                        for (int k = 0; k < WAVE; k++) {
                            const double px = C.x[lane + k], py = C.y[lane + k], pz = C.z[lane + k];
                            const int ptf = C.tf[lane + k];
                            const int pfl = ptf >> 16;
                            const int p = ((lane + k) & (WAVE - 1)) + WAVE * q;   // slot in tile J
                            double psr = 0.0, prr = 0.0, pq = 0.0;
                            int pix = 0;
                            if constexpr (RF) {
                                psr = C.sr[lane + k]; prr = C.rg[lane + k]; pq = C.q[lane + k];
                                pix = C.ix[lane + k];
                            }
                            double hx = 0.0, hy = 0.0, hz = 0.0;    // pair force on the partner (negated)
#pragma unroll
                            for (int u = 0; u < TPL; u++) {
                                const int tfl = ttf[u] >> 16;
                                const int both = tfl & pfl;
                                bool skip = !(both & SL_VALID) || (both & (SL_SITE | SL_FIXED)) ||
                                            (diag && p <= lane + WAVE * u);
                                const double dx = tx[u] - px, dy = ty[u] - py, dz = tz[u] - pz;
                                double d2 = dx * dx + dy * dy + dz * dz;
                                d2 = skip ? 1e30 : d2;
                                const bool mx = ((tfl | pfl) & SL_SITE) != 0;   // a site: no reaction field
                                if constexpr (PAIRS) {
                                    const double4 tl = make_double4(pr.sc3, pr.fct, pr.dm2hi, 0.0);
                                    double y, de;
                                    if (TAB || (pr.flags & PF_EFPOT)) {
                                        de = pair_near_far(pr, tl, P.ep, P.ires, d2, y);
                                        if constexpr (EN) sum2_add(e0, skip ? 0.0 : y);
                                    } else {
                                        double q0 = 0.0, q1 = 0.0, q2 = 0.0;
                                        de = pair_analytic(pr, P, d2, q0, q1, q2);
                                        if constexpr (EN) {
                                            sum2_add(e1, skip ? 0.0 : q0);
                                            sum2_add(e2, skip ? 0.0 : q1);
                                            sum2_add(e3, skip ? 0.0 : q2);
                                        }
                                    }
                                    de = skip ? 0.0 : de;
                                    const double fxp = de * dx, fyp = de * dy, fzp = de * dz;
                                    if (tfl & SL_RECV) { ax_[u] += fxp; ay_[u] += fyp; az_[u] += fzp; }
                                    hx += fxp; hy += fyp; hz += fzp;
                                }
                                if constexpr (RF) {
                                    // rfpar.f90:177-223 for the ion pair (lo, hi) by index: counted when
                                    // srfe(lo) is nonzero and hi is moving and inside the grid box
                                    const bool thi = tix[u] > pix;
                                    const bool on = !skip && !mx &&
                                                    (thi ? (psr != 0.0 && (tfl & SL_HI)) : (tsr[u] != 0.0 && (pfl & SL_HI)));
                                    const double m = on ? 1.0 : 0.0;
                                    const double aux0 = P.celec * tq[u] * pq;
                                    const double srfeij = tsr[u] * psr, reffij = trr[u] * prr;
                                    const double rfdn = rsqrt_s26(reffij * reffij + (on ? d2 : 1.0));
                                    const double rfcf = reffij * rfdn;
                                    const double aux1 = aux0 * rfcf;
                                    const double aux2 = aux0 * srfeij * (rfdn * (rfdn * rfdn));
                                    const double aux3 = -aux2 * ((on ? d2 : 1.0) + reffij * 0.5);
                                    const double der = m * (aux2 * reffij);
                                    if constexpr (EN) sum2_add(erf, m * (aux1 * srfeij));
                                    aa_[u] = fma(m, -aux1 * psr, aa_[u]);
                                    ab_[u] = fma(m, aux3 * prr, ab_[u]);
                                    ga = fma(m, -aux1 * tsr[u], ga);
                                    gb = fma(m, aux3 * trr[u], gb);
                                    ax_[u] = fma(der, dx, ax_[u]);
                                    ay_[u] = fma(der, dy, ay_[u]);
                                    az_[u] = fma(der, dz, az_[u]);
                                    gx = fma(-der, dx, gx);
                                    gy = fma(-der, dy, gy);
                                    gz = fma(-der, dz, gz);
                                }
                            }
                            if constexpr (PAIRS) {
                                const double pw = (pfl & SL_RECV) ? 1.0 : 0.0;
                                gx -= pw * hx; gy -= pw * hy; gz -= pw * hz;
                            }
                            gx = wave_next(gx); gy = wave_next(gy); gz = wave_next(gz);
                            if constexpr (RF) { ga = wave_next(ga); gb = wave_next(gb); }
                        }
                    };
                    if (!fast) general(std::true_type{});
                    else if constexpr (RF) general(std::false_type{});
                }
                // the next chunk's staging stays below this chunk's reads
                __atomic_signal_fence(__ATOMIC_SEQ_CST);
            }
            rfany |= rfsums;
            if (diag) {   // partner sums of the tile's own slots
#pragma unroll
                for (int u = 0; u < TPL; u++) {
                    if (u != q) continue;
                    ax_[u] += gx; ay_[u] += gy; az_[u] += gz;
                    if constexpr (RF) { aa_[u] += ga; ab_[u] += gb; }
                }
            } else {
                // a chunk without reaction-field sums writes the three force components only
                // and says so in its flag, which k_tfin reads before it reads the A and B rows
                double *const dp = prow + WAVE * q + lane;
                dp[0] = gx; dp[(size_t)TT] = gy; dp[2 * (size_t)TT] = gz;
                if constexpr (RF) {
                    if (rfsums) { dp[3 * (size_t)TT] = ga; dp[4 * (size_t)TT] = gb; }
                    if (lane == 0) pflag[q] = rfsums ? 1 : 0;
                }
            }
        }
    }
    // the item's row of tile I: after its I partner rows, one per group from I's own
    const size_t trow = (size_t)tile_row(I, n, R) + I + (g - I / R);
    double *const dst = P.tpart + trow * NC * TT + lane;
#pragma unroll
    for (int u = 0; u < TPL; u++) {
        // the fast sweeps add to every target, a site that is not free too
        const int f = ttf[u] >> 16;
        const bool keep = (f & (SL_SITE | SL_RECV)) != SL_SITE;
        double *const d = dst + WAVE * u;
        d[0] = keep ? ax_[u] : 0.0; d[(size_t)TT] = keep ? ay_[u] : 0.0; d[2 * (size_t)TT] = keep ? az_[u] : 0.0;
        if constexpr (RF) {
            if (rfany) {
                d[3 * (size_t)TT] = (f & SL_RFON) ? fma(-P.celec * tq[u], wa[u], aa_[u]) : aa_[u];
                d[4 * (size_t)TT] = ab_[u] - wb[u];
            }
            if (lane == 0) P.tflag[trow * TPL + u] = rfany ? 1 : 0;
        }
    }
    if constexpr (EN) {
        if (eclass >= 0) ener_end(eclass);
        ener_out(TE_RFPAR, erf);
        if (lane == 0) {   // the classes the item has no pair of
            if (!(edone & 1)) { ener_zero(TE_EFPOT); ener_zero(TE_ELEC); ener_zero(TE_VDW); ener_zero(TE_SRPMF); }
            if (!(edone & 2)) { ener_zero(TE_EFPOTMX); ener_zero(TE_QQMX); ener_zero(TE_VDWMX); ener_zero(TE_SRPMFMX); }
        }
    }
}

// sum over the 8 lanes of a group (lanes 8g..8g+7); every lane gets the same bits
__device__ __forceinline__ double group8_sum(double v) {
    v += __shfl_xor(v, 1, WAVE);
    v += __shfl_xor(v, 2, WAVE);
    v += __shfl_xor(v, 4, WAVE);
    return v;
}

// k_tfin: slot s of the tile order, eight lanes per slot (32 slots per block).  The
// lanes split the slot's partial rows -- rows of one type pull one way and those of the next
// the other, so the sums carry their rounding errors -- then its grid corners (lane c takes
// corner c of the trilinear stencils, c, c + 8, .. of the 27-node B-spline); lane 0 of the
// group finishes the particle.  Sites and moving ions are finished as by k_step; a fixed ion
// only receives its reaction-field force (rfpar.f90:177-223 applies it to both ions of a
// pair), written when forces are asked for.
template <int FEAT>
__global__ __launch_bounds__(BLOCK) void k_tfin(StepParams P) {
    constexpr bool RF = (FEAT & F_RFT) != 0;
    const int tid = threadIdx.x, sub = tid & 7;
    const int s = blockIdx.x * (BLOCK / 8) + (tid >> 3);
    const int nslot = P.ntile * WAVE * P.ttpl, ss = s < nslot ? s : 0;
    const double4 pa = P.spos[ss];
    const bool sv = s < nslot && __double2hiint(pa.w) >= 0;   // else an empty slot
    const int i = sv ? __double2hiint(pa.w) : 0, t2 = __double2loint(pa.w);
    const int ns = P.nsites;
    const bool is_site = i < ns, fixed = !is_site && i < ns + P.nfix;
    const int TT = WAVE * P.ttpl, n = P.ntile, NC = RF ? 5 : 3, R = P.trun;
    const int I = ss / TT, t = ss - I * TT;
    Sum2 sum[5] = {};
    // the slot's rows: one per lower tile, one per column group from its own; rows K = sub,
    // sub + 8, .. added in that order, KU of them per iteration so that their
    // loads (the flags, then the rows) are in flight together
    constexpr int KU = 8;
    const size_t row0 = (size_t)tile_row(I, n, R);
    const int nrow = (int)(tile_row(I + 1, n, R) - row0);
    for (int K0 = sub; K0 < nrow; K0 += 8 * KU) {
        bool ok[KU], ab[KU];
        const double *src[KU];
#pragma unroll
        for (int u = 0; u < KU; u++) {
            const int K = K0 + 8 * u;
            ok[u] = K < nrow;
            const size_t row = row0 + (ok[u] ? K : 0);
            src[u] = P.tpart + row * NC * TT + t;
            ab[u] = false;
            // the A and B rows only where they were written
            if constexpr (RF) {
                const int32_t fl = P.tflag[row * P.ttpl + (t >> 6)];
                ab[u] = ok[u] & (fl != 0);
            }
        }
        double r[KU][5];
#pragma unroll
        for (int u = 0; u < KU; u++) {
#pragma unroll
            for (int c = 0; c < 3; c++) r[u][c] = src[u][(size_t)c * TT];
            r[u][3] = r[u][4] = 0.0;
            if constexpr (RF) {
                if (ab[u]) { r[u][3] = src[u][3 * (size_t)TT]; r[u][4] = src[u][4 * (size_t)TT]; }
            }
        }
        // KU rows plainly, their sum with its rounding error: no slower than plain sums (row by
        // row that took 0.12 ms more of 3 at 56,000 particles)
#pragma unroll
        for (int c = 0; c < NC; c++) {
            double v = 0.0;
#pragma unroll
            for (int u = 0; u < KU; u++)
                if (ok[u] && (c < 3 || ab[u])) v += r[u][c];
            sum2_add(sum[c], v);
        }
    }
    double acc[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int c = 0; c < NC; c++) {
        const Sum2 t = group_sum2<8>(sum[c]);
        acc[c] = isfinite(t.s) ? t.s + t.c : t.s;   // the error of an infinite sum is not a number
    }

    // grids of a target (a site or a moving ion): staticf1.f90:45-118, vdwgd1trln.f90:
    // 50-161 / vdwgd1spln.f90:50-170, corners split over the group's lanes
    double gfx = 0.0, gfy = 0.0, gfz = 0.0, egx = 0.0, egv = 0.0, ph = 0.0;
    bool vin = false;
    const bool target = sv && !fixed;
    if constexpr ((FEAT & F_PHIX) != 0) {
        const GridGeom &g = P.gx;
        double chi;
        bool ok;
        if (is_site) { ok = P.namsite[i] == 1; chi = P.cgnuc; }
        else { ok = true; chi = P.cg[abs(P.typei[i])]; }
        ok = ok && target && pa.x <= g.xbcen + g.tranx && pa.x >= g.xbcen - g.tranx &&
             pa.y <= g.ybcen + g.trany && pa.y >= g.ybcen - g.trany &&
             pa.z <= g.zbcen + g.tranz && pa.z >= g.zbcen - g.tranz;
        if (ok) {
            double xi, yi, zi;
            int ix, iy, iz;
            grid_cell(g, pa.x, pa.y, pa.z, xi, yi, zi, ix, iy, iz);
            double e = 0.0;
            tri_corner(g, P.phix, xi, yi, zi, ix, iy, iz, sub, P.celec * chi, gfx, gfy, gfz, e);
            egx += e;
        }
    }
    if constexpr ((FEAT & F_PHIV) != 0) {
        const GridGeom &g = P.gv;
        const int8_t *phiv = P.phiv + vdw_map_of(P, i);
        double esvdw = P.svdw;
        if (P.flags & QSVDW) esvdw = P.svdw * P.scal[t2];
        if (P.flags & QBSPLINE) {
            vin = target && pa.x <= g.xbcen + g.tranx - g.dcel && pa.x >= g.xbcen - g.tranx + g.dcel &&
                  pa.y <= g.ybcen + g.trany - g.dcel && pa.y >= g.ybcen - g.trany + g.dcel &&
                  pa.z <= P.vzmax && pa.z >= P.vzmin;
            if (vin) {
                double xi, yi, zi;
                int ix, iy, iz;
                spline_cell(g, pa.x, pa.y, pa.z, xi, yi, zi, ix, iy, iz);
                for (int c = sub; c < 27; c += 8) {
                    const int k = ix - 1 + c / 9, l = iy - 1 + (c / 3) % 3, m = iz - 1 + c % 3;
                    double ai, dai, bi, dbi, ci, dci;
                    bspline_m3(1.5 - (xi - k * g.dcel) * g.idcel, ai, dai);
                    bspline_m3(1.5 - (yi - l * g.dcel) * g.idcel, bi, dbi);
                    bspline_m3(1.5 - (zi - m * g.dcel) * g.idcel, ci, dci);
                    if ((ai != 0.0 || dai != 0.0) && (bi != 0.0 || dbi != 0.0) &&
                        (ci != 0.0 || dci != 0.0)) {
                        const double v = (double)phiv[((size_t)k * g.ny + l) * g.nz + m];
                        ph += v;
                        const double phivsv = v * esvdw;
                        const double prefac = phivsv * g.idcel;
                        gfx += dai * bi * ci * prefac;
                        gfy += ai * dbi * ci * prefac;
                        gfz += ai * bi * dci * prefac;
                        egv += ai * bi * ci * phivsv;
                    }
                }
            }
        } else {
            vin = target && pa.x <= g.xbcen + g.tranx && pa.x >= g.xbcen - g.tranx &&
                  pa.y <= g.ybcen + g.trany && pa.y >= g.ybcen - g.trany && pa.z <= P.vzmax &&
                  pa.z >= P.vzmin;
            if (vin) {
                double xi, yi, zi;
                int ix, iy, iz;
                grid_cell(g, pa.x, pa.y, pa.z, xi, yi, zi, ix, iy, iz);
                ph = tri_corner(g, phiv, xi, yi, zi, ix, iy, iz, sub, esvdw, gfx, gfy, gfz, egv);
            }
        }
    }
    gfx = group8_sum(gfx);
    gfy = group8_sum(gfy);
    gfz = group8_sum(gfz);
    if (P.write_energy) {
        egx = group8_sum(egx);
        egv = group8_sum(egv);
    }
    ph = group8_sum(ph);   // map values are integers: exact in any order
    if (sub != 0 || !sv) return;

    if (fixed) {
        if constexpr (RF) {
            if (P.write_forces) {
                double f[3] = {0.0, 0.0, 0.0};
                if (P.rfa[i].z != 0.0) {
                    const double4 dst = P.rfd[2 * (size_t)i], drt = P.rfd[2 * (size_t)i + 1];
                    f[0] = acc[0] + acc[3] * dst.x + acc[4] * drt.x;
                    f[1] = acc[1] + acc[3] * dst.y + acc[4] * drt.y;
                    f[2] = acc[2] + acc[3] * dst.z + acc[4] * drt.z;
                }
                P.fx[i] = f[0]; P.fy[i] = f[1]; P.fz[i] = f[2];
            }
        }
        return;
    }
    double F[3] = {acc[0] + gfx, acc[1] + gfy, acc[2] + gfz};
    double erf_self = 0.0;
    if constexpr (RF) {
        if (!is_site) {
            // the self term of a moving ion (rfpar.f90:146-156) and the variation of its
            // srfe and reff in every pair (A, B summed over the tile pairs)
            const double4 ra = P.rfa[i];
            if (ra.z != 0.0) {
                const double4 dst = P.rfd[2 * (size_t)i], drt = P.rfd[2 * (size_t)i + 1];
                const double cgt = P.cg[abs(P.typei[i])];
                const double aux = P.celec * cgt * cgt * ra.x;
                const double a_s = acc[3] - aux;
                F[0] += a_s * dst.x + acc[4] * drt.x;
                F[1] += a_s * dst.y + acc[4] * drt.y;
                F[2] += a_s * dst.z + acc[4] * drt.z;
                erf_self = 0.5 * aux * ra.x;
            }
        }
    }
    if constexpr ((FEAT & F_DNA) != 0) {
        if (is_site) {
            const double4 fd = P.fdna[i];   // CG-DNA list terms from k_dna
            F[0] += fd.x; F[1] += fd.y; F[2] += fd.z;
        }
    }
    if (P.mmon && !is_site) {   // MMIJ reaction field (k_mm_force)
        const double4 fr = P.frf[i];
        F[0] += fr.x; F[1] += fr.y; F[2] += fr.z;
    }
    const bool warned = vin && ph >= ((P.flags & QBSPLINE) ? P.thold27 : P.thold8);
    if (warned) atomicAdd(&P.warn[t2], 1);
    if (P.flags & QMEMB) {   // MEMBRANE, membrane.f90:36-104
        const double chg = is_site ? (P.namsite[i] == 1 ? P.cgnuc : 0.0) : P.cg[abs(P.typei[i])];
        bool mw;
        const double em = membrane_energy(P, pa.x, pa.y, pa.z, chg, t2, F, mw);
        if (mw) atomicAdd(&P.warn[t2], 1);
        if (P.write_energy) P.epart[(size_t)E_MEMB * P.ecap + i] = em;
    }
    if (P.write_energy) {
        // the pair categories are summed per tile pair (tener); the grid and reaction-field
        // self terms per particle
        double *ep_ = P.epart + i;
        const size_t cs = P.ecap;
        ep_[E_GSBPA * cs] = egx;
        ep_[E_VDWGD * cs] = egv;
        if (is_site) {
            ep_[E_EFPOTMX * cs] = 0.0; ep_[E_QQMX * cs] = 0.0;
            ep_[E_VDWMX * cs] = 0.0; ep_[E_SRPMFMX * cs] = 0.0;
        } else {
            ep_[E_EFPOT * cs] = 0.0; ep_[E_ELEC * cs] = 0.0;
            ep_[E_VDW * cs] = 0.0; ep_[E_SRPMF * cs] = 0.0;
            if constexpr (RF) ep_[E_RFPAR * cs] = erf_self;
        }
    }
    if (P.write_forces) {
        P.fx[i] = F[0];
        P.fy[i] = F[1];
        P.fz[i] = F[2];
    }
    if constexpr ((FEAT & F_UPDATE) != 0) {
        if (P.vacc) P.vacc[i] += F[0] * pa.x + F[1] * pa.y + F[2] * pa.z;
        const bool fr = !is_site || ((FEAT & F_DNA) && P.stfree[i] != 0);
        if (!fr) {
            P.poso[i] = pa;
            P.sposo[s] = pa;
            return;
        }
        const double4 pn = bd_update(P, i, is_site, pa, F, noise_row(P, i));
        P.poso[i] = pn;
        P.sposo[s] = pn;
    }
}

template <int FEAT>
static void dispatch_tiles(const StepParams &p, hipStream_t s, int which) {
    constexpr int TF = FEAT & (F_DNA | F_TAB | F_RFT);
    if (which & 1) {
        const dim3 grid(p.titems), block(WAVE);
#define TILES(T)                                                                          \
    do {                                                                                  \
        if (p.write_energy) hipLaunchKernelGGL((k_tiles<TF, T, true>), grid, block, 0, s, p); \
        else hipLaunchKernelGGL((k_tiles<TF, T, false>), grid, block, 0, s, p);           \
    } while (0)
        switch (p.ttpl) {
            case 1: TILES(1); break;
            case 2: TILES(2); break;
            default: TILES(4); break;
        }
#undef TILES
    }
    if (which & 2)
        hipLaunchKernelGGL((k_tfin<FEAT & ~F_TAB>), dim3((p.ntile * WAVE * p.ttpl + BLOCK / 8 - 1) / (BLOCK / 8)),
                           dim3(BLOCK), 0, s, p);
}

hipError_t launch_tiles(const StepParams &p, hipStream_t s, int which) {
    if (p.ntot <= 0) return hipSuccess;
    int feat = 0;
    if (p.flags & QNUCL) feat |= F_DNA;
    if (p.flags & QPHIX) feat |= F_PHIX;
    if (p.flags & QPHIV) feat |= F_PHIV;
    if (p.mode == 1) feat |= F_UPDATE;
    if (p.all_efpot) feat |= F_TAB;
    if (p.rfon) feat |= F_RFT;
#define CASE(F) case F: dispatch_tiles<F>(p, s, which); break;
    switch (feat) {
        CASE(0) CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7)
        CASE(8) CASE(9) CASE(10) CASE(11) CASE(12) CASE(13) CASE(14) CASE(15)
        CASE(16) CASE(17) CASE(18) CASE(19) CASE(20) CASE(21) CASE(22) CASE(23)
        CASE(24) CASE(25) CASE(26) CASE(27) CASE(28) CASE(29) CASE(30) CASE(31)
        CASE(64) CASE(65) CASE(66) CASE(67) CASE(68) CASE(69) CASE(70) CASE(71)
        CASE(72) CASE(73) CASE(74) CASE(75) CASE(76) CASE(77) CASE(78) CASE(79)
        CASE(80) CASE(81) CASE(82) CASE(83) CASE(84) CASE(85) CASE(86) CASE(87)
        CASE(88) CASE(89) CASE(90) CASE(91) CASE(92) CASE(93) CASE(94) CASE(95)
    }
#undef CASE
    return hipGetLastError();
}

}  // namespace bromoc
