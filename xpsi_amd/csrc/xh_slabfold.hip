// Slab fold: the moment form of the cell x phase x energy spline fold with its
// operands formed once per block and handed to the matrix cores through LDS.
//
// Reference behaviour: the energy x cell x phase spline loop of
// xpsi/cellmesh/integrator_for_azimuthal_invariance.pyx:565-596 with the
// blackbody intensity of xpsi/surface_radiation_field/hot_BB.pyx:54-98 or the
// 4-D table of hot_Num4D.pyx:248-438.  As in k_moment_fold (xh_moment.hip),
// where the periodic Akima piece s_k of energy k is >= 0 over its interval i
//
//     sum_j A_j s_k(x_jp) = sum_i sum_m coef_k[i][m] * MOM[i][m][p],
//
// one 16x16x4 product per interval, 16 energies and 16 phases; pieces <= 0
// throughout fold nothing and sign-changing pieces are evaluated cell by cell
// with the reference's clipping.
//
// A block of 4 EC wavefronts owns one member, 64 EC energies, 64 phases and a
// few parallels.  A parallel and image's intervals are taken in slabs: RUN
// successive intervals of each quarter of the turn.  Between two barriers every
// wavefront forms its share of the next slab's operands and folds this slab's:
//   operands  the Akima pieces of 64 energies over its quarter's RUN intervals
//             (lanes = energies; profile, secants and slopes in a window that
//             slides through the quarter in registers) and the cell moments of 64
//             phases over one interval or two (lanes = phases), into one of two
//             LDS buffers in the order of the products' operands;
//   products  its own 64 energies x 16 phases over the slab's intervals (one
//             16-byte and one 4-byte LDS read per interval for four products),
//             then the sign-changing pieces cell by cell, evaluated by the
//             same product (coefficients x powers of the cells' offsets).
// Half of the wavefronts begin with the operands and half with the products.
//
// Why this split.  A 64 x 64 tile and interval is 16 products, about 85 vector
// instructions for the pieces of 64 energies and about 130 for the moments of 64
// phases.  A wavefront that forms both for its own tile (k_wave_fold) is bound
// by them, by sign-changing pieces taken one energy at a time and by the
// atomics of its short FP32 chains; blocks of one parallel's whole interval list
// (k_moment_fold) by their set-up and barriers.  Here the moments serve EC
// chunks and the pieces four phase tiles; a run of full cells on an evenly
// spaced parallel has its moments in closed form; a tile skips the intervals
// that none of its phases reaches (a spot covers part of the turn); and as a
// slab holds intervals of every quarter, the tiles of a narrow spot still have
// like work between barriers (slabs of 16 successive intervals were 1.46 times as
// slow, on 1100 members with FP64 products).  Bound now by the first reads of each
// parallel and by vector issue (operands): of the wavefronts' time on 1100
// members at 256 energies 37% are a parallel's first reads, 14% the wait for the
// other wavefronts' reads, 15% its set-up, 13% the operands, 10% the slabs' barriers and 7%
// the products; on eight large members (256 leaves, 512 energies) 22, 2, 8, 30, 21
// and 15%.  Measured, fold alone, ms (before: the automatic choice then):
//   1100 blackbody members of 24 to 96 cells a side, 64 leaves and phases, 256
//     energies, FP32                                  27.1 (k_wave_fold) -> 19.2
//   512 of them, 128 energies, FP32                    7.04 (k_wave_fold) -> 4.7
//   128 members of 16 to 64 cells, 128 energies, FP64  10.0 (k_moment_fold) -> 1.4
//   one member, 32 cells, 128 energies, FP64           0.070 (k_moment_fold) -> 0.039
//   192 requests of 4 table members, 128 leaves and phases, 256 energies, FP32
//     79.2 (k_moment_fold with the intensities formed in it) -> 15.9 (profiles included)
//   4 table members, FP64                              2.96 -> 0.60
//
// Accumulation.  In the FP32 form a slab's products of one tile (at most eight
// intervals) are one FP32 chain from zero on v_mfma_f32_16x16x4f32, added to
// FP64 sums in registers times the parallel's reference cell area; the tiles
// are taken in two pairs, so that the chains need eight registers beside the 32
// of the sums (all four at once spilled).  FP64 products throughout (64 cycles
// of the matrix unit where these take 32) were 1.06 times as slow (1100
// members), with 0.6 of this form's flux error.  A wavefront's sums stay in registers
// over all its parallels and reach the flux with one FP64 atomic per entry.
//
// Precision of the blackbody profile.  I = E^3 G / (exp(E' / kT) - 1) with
// E' = E / Z: the factor E^3 is common to all knots of an energy and is applied
// in FP64 with the final scale, G = geometric factor / Z^3 is formed in FP64
// and rounded once, and the exponent is reduced in FP64 before the FP32
// exponential, so its relative error does not grow with E' / kT.  Flux of the
// precision form against FP64 (2-norm): 3.5e-9 to 5.4e-9 (k_wave_fold: 9e-9 to
// 1.2e-8).
#include <limits.h>
#include "xh_common.hpp"
#include "xh_types.hpp"
#include "xh_kernels.hpp"
#include "xh_atm.hpp"
#include "xh_fold.hpp"

namespace xh {

namespace {

constexpr double LOG2E = 1.4426950408889634074;

// 2^60 / (2^t - 1), t reduced in FP64; zero where 2^t leaves the FP32 range.
// The power of two keeps every nonzero value, the secants and the pieces far
// from the denormals, where a piece's sign class would have to be settled by
// its extremes (and often as sign-changing) for every energy of a cold spot.
constexpr double PROFILE_UNIT = 0x1p60, TABLE_UNIT = 0x1p40;   // TABLE_UNIT: the same for the table's profile
__device__ __forceinline__ float planck_factor(double t, float)
{
    const double n = __builtin_rint(t);
    const float f = (float)(t - n);
    const float d = __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(f), (int)fmin(n, 200.0) - 60) - 0x1p-60f;
    // reciprocal with two Newton steps
    float r = __builtin_amdgcn_rcpf(d);
    r = fmaf(fmaf(-d, r, 1.0f), r, r);
    r = fmaf(fmaf(-d, r, 1.0f), r, r);
    return t < 127.5 ? r : 0.0f;
}
__device__ __forceinline__ double planck_factor(double t, double) { return 1.0 / (exp(t) - 1.0); }

// t's unit in planck_factor: log2 e / kT for FP32, 1 / kT for FP64
template <typename R> struct TUnit { static constexpr double v = 1.0; };
template <> struct TUnit<float> { static constexpr double v = LOG2E; };

__device__ __forceinline__ float quot(float a, float b)
{
    float r = __builtin_amdgcn_rcpf(b);
    r = fmaf(fmaf(-b, r, 1.0f), r, r);
    const float q = a * r;
    return fmaf(fmaf(-b, q, a), r, q);
}
__device__ __forceinline__ double quot(double a, double b) { return a / b; }

// cubic_class (xh_fold.hpp: same classes, same margin) of a piece whose
// Bernstein points leave its sign open, as a cubic in t / h relative to the sum
// of its terms: the discriminant cannot leave the FP32 range, whatever the unit
template <typename R>
__device__ __forceinline__ int open_class(R a, R b, R c, R d, R h)
{
    b *= h;
    c *= h * h;
    d *= h * h * h;
    const R r = (R)1 / (fabs(a) + fabs(b) + fabs(c) + fabs(d));
    a *= r; b *= r; c *= r; d *= r;
    const R tol = (R)64 * Eps<R>::v, b3 = a + b + c + d;
    const R b1 = a + b * (R)(1.0 / 3.0), b2 = a + ((R)2 * b + c) * (R)(1.0 / 3.0);
    R lo = fmin(fmin(a, b1), fmin(b2, b3)), hi = fmax(fmax(a, b1), fmax(b2, b3));
    if (lo >= -tol) return 1;
    if (hi <= tol) return 0;
    auto f = [&](R t) { return a + t * (b + t * (c + t * d)); };
    lo = fmin(a, b3);
    hi = fmax(a, b3);
    R r1 = (R)-1, r2 = (R)-1;
    if (d != (R)0) {
        const R disc = c * c - (R)3 * b * d;
        if (disc >= (R)0) {
            const R q = -(c + copysign(sqrt(disc), c));
            if (q != (R)0) { r1 = q / ((R)3 * d); r2 = b / q; }
            else r1 = (R)0;
        }
    } else if (c != (R)0) r1 = -b / ((R)2 * c);
    if (r1 > (R)0 && r1 < (R)1) { const R v = f(r1); lo = fmin(lo, v); hi = fmax(hi, v); }
    if (r2 > (R)0 && r2 < (R)1) { const R v = f(r2); lo = fmin(lo, v); hi = fmax(hi, v); }
    if (lo >= -tol) return 1;
    if (hi <= tol) return 0;
    return 2;
}

// a value that the compiler takes as new: what is formed from it (operand
// addresses, above all) is formed where it is used and not held in registers
// across the stages
__device__ __forceinline__ int fresh(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

}  // namespace

// grid: x = (ring block, slab range), y = energy chunk x phase chunk, z = member;
// 256 EC threads; dynamic LDS slab_fold_lds(...).  The flux is zeroed beforehand.
template <typename R, int ATM, int EC>
__global__ void __launch_bounds__(256 * EC, 4) k_slab_fold(const Member* __restrict__ members, Layout L, FoldArgs F)
{
    constexpr int NW = 4 * EC, NT = 64 * NW;
    constexpr int RUN = slab_run(sizeof(R)), SL = 4 * RUN;   // intervals of a wavefront's coefficients; of a slab
    constexpr int MRUN = SL > NW ? SL / NW : 1;   // intervals of a wavefront's moments (of the first SL / MRUN wavefronts)
    typedef typename Mfma<double>::v4 v4;
    const int mi = blockIdx.z, tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // scalar: its indexes and branches stay off the vector units
    const Member& m = members[mi];
    if (!m.active || m.status) return;
    if (ATM == 2 && *F.item_total <= F.pass * F.cap) return;
    const int S = m.S, correct = m.correct;
    const int N_L = L.N_L, N_P = L.N_P, N_E = L.N_E, NI = N_L - 1;
    // a member has fewer parallels than the grid's bound: its blocks are taken
    // in a turn of its own, so that the empty ones do not fall on the same XCDs
    const int bx = (blockIdx.x + blockIdx.z) % gridDim.x;
    const int r0 = (bx / F.splits) * F.ring_block;
    if (r0 >= S) return;
    const int r1 = min(S, r0 + F.ring_block);
    const int Q = (NI + 3) >> 2, n_slab = (Q + RUN - 1) / RUN, sp = bx % F.splits;
    const int s_begin = sp * n_slab / F.splits, s_end = (sp + 1) * n_slab / F.splits;
    if (s_begin >= s_end) return;
    const int n_pc = (N_P + 63) >> 6;
    const int e0 = (blockIdx.y / n_pc) * (64 * EC), p0 = (blockIdx.y % n_pc) * 64;

    // parts of fixed size first, so that only the last two need their offsets kept
    extern __shared__ __align__(16) double ssm[];
    R* CO = (R*)ssm;                          // [2][SL][EC][64][4]: lane (power m, energy % 16), chunk of 16 energies
    R* MOM = CO + 2 * SL * EC * 256;          // [2][SL][4][64]: phase tile, lane (power m, phase % 16)
    unsigned long long* MASK = (unsigned long long*)(MOM + 2 * SL * 256);   // [2][SL] phases with cells
    unsigned long long* ANZ = MASK + 2 * SL;  // [2][SL][EC] energies with a product term
    unsigned long long* MIXM = ANZ + 2 * SL * EC;   // [2][SL][EC] energies whose piece changes sign
    double* AM = (double*)(MIXM + 2 * SL * EC);     // [8] a wavefront's largest area
    SlabPhase* PL = (SlabPhase*)(AM + 8);     // [64] a phase's turn of the cells
    int* CF = (int*)(PL + 64);                // [2][SL][64] first cell | cells << 16 of a phase in an interval
    int* AF = CF + 2 * SL * 64;               // [8] a wavefront's flags on the cells' azimuths
    SlabKnot<R>* KN = (SlabKnot<R>*)(AF + 8); // [N_L]
    SlabCell<R>* CELL = (SlabCell<R>*)(KN + N_L);   // [S_max]

    // roles: wavefront w forms the pieces of energy chunk ec over quarter rq of
    // the turn and folds chunk ec x phase tile rq; lane = energy or phase
    const int ec = w % EC, rq = w / EC;
    const int e = e0 + 64 * ec + lane;
    const bool chunk_on = e0 + 64 * ec < N_E, e_ok = e < N_E;
    const double E = F.energies[min(e, N_E - 1)];
    const int pc = p0 + 16 * rq + (lane & 15);          // the phase this lane folds
    const bool tile_on = chunk_on && p0 + 16 * rq < N_P;
    const double php = p0 + lane < N_P ? F.phases[p0 + lane] : 0.0;   // the phase whose moments it forms
    const int np = p0 + lane < N_P ? S : 0;
    const double phc = pc < N_P ? F.phases[pc] : 0.0;

    v4 acc[4];
#pragma unroll
    for (int c = 0; c < 4; c++) acc[c] = v4{0.0, 0.0, 0.0, 0.0};
    const size_t cbase = (size_t)mi * L.S_max * L.S_max;
    const double* phis = F.phi + (size_t)mi * L.S_max * (F.phi_row_stride ? L.S_max : 1);

    double logT_in = __builtin_nan(""), kT = 1.0, x_else = 0.0;
    double a_ref = 1.0, invd = 0.0;
    int order = 0;                                      // of the parallel's azimuths: 0 none, 1 increasing, 2 evenly spaced
    // a parallel's images (a lane each), read one parallel ahead: an image's first
    // reads wait for no other (read with each image, a parallel waited twice:
    // 1100 members 0.2 ms, 8 walkers 0.175 -> 0.171 ms)
    auto shown = [&](int i) -> int { return lane < L.IO_max ? F.valid[((size_t)mi * L.S_max + i) * L.IO_max + lane] : 0; };
    int v_next = shown(r0);
    for (int i = r0; i < r1; i++) {
        const size_t ro = (size_t)mi * L.S_max + i;
        const unsigned long long seen = __ballot(v_next != 0);
        const int images = ~seen ? __builtin_ctzll(~seen) : 64;
        if (i + 1 < r1) v_next = shown(i + 1);
        long long slot0 = 0;                            // table: the parallel's first profile
        if (ATM == 2) {
            slot0 = (long long)F.item0[ro] - (long long)F.pass * F.cap;
            if (slot0 < 0 || slot0 >= F.cap) continue;  // another pass's
        }
        for (int I = 0; I < images; I++) {
            const R* prof = ATM == 2 ? (const R*)F.prof + (size_t)(slot0 + I) * N_L * N_E + min(e, N_E - 1) : nullptr;
            // everything read from memory for this parallel and image at once
            const size_t vix = ro * L.IO_max + I;
            const double* g = F.geo + vix * 5 * N_L;
            const double* area = F.cellArea + cbase + (size_t)i * S;
            const int* radp = F.radiates ? F.radiates + cbase + (size_t)i * S : nullptr;
            const double* prow = phis + (size_t)i * F.phi_row_stride;
            const double last_q = g[5 * N_L - 1];
            double gq[4] = {0.0, 1.0, 0.0, 0.0}, g_next = 0.0, gz0 = 1.0, gg0 = 0.0, gp0 = 0.0;
            if (tid < N_L) {
#pragma unroll
                for (int k = 0; k < 4; k++) gq[k] = g[(k < 2 ? k : k + 1) * N_L + tid];   // PHASE, Z, GEOM, PREV
                if (tid < NI) g_next = g[tid + 1];
                else { gz0 = g[N_L]; gg0 = g[3 * N_L]; gp0 = g[4 * N_L]; }
            }
            double ca = 0.0, cp = 0.0, cp1 = 0.0, cp_first = 0.0, cp_last = 0.0;
            bool cr = false;
            if (I == 0 && tid < S) {
                ca = area[tid];
                cr = radp ? radp[tid] == 1 : ca > 0.0;
                cp = prow[tid];
                cp1 = prow[min(tid + 1, S - 1)];
                cp_first = prow[0];
                cp_last = prow[S - 1];
            }
            const double logT = F.logT[ro];
            // the next parallel's geometry and cells are touched now, so that
            // they come from the L2 cache when their turn comes
            double touch = 0.0;
            if (i + 1 < r1) {
                const int q = tid - 5 * N_L;
                touch = q < 0 ? (g + (size_t)L.IO_max * 5 * N_L)[tid] : (q < S ? area[S + q] : 0.0);
            }
            if (ATM == 1 && logT != logT_in) {
                logT_in = logT;
                kT = K_B_OVER_KEV * pow(10.0, logT);
                x_else = kT / (K_B_OVER_KEV * pow(10.0, m.else_logT));   // t of the elsewhere temperature / t
            }
            __syncthreads();                            // the previous image's reads are done
            // the last leaf repeats the first when it was not queried itself
            const bool copy_last = last_q < -1.0;
            for (int q = tid; q < N_L; q += NT) {
                double x = gq[0], z = gq[1], geom = gq[2], pq = gq[3], xn = g_next;
                if (q != tid) {
                    x = g[q]; z = g[N_L + q]; geom = g[3 * N_L + q]; pq = g[4 * N_L + q];
                    if (q < NI) xn = g[q + 1];
                    else { gz0 = g[N_L]; gg0 = g[3 * N_L]; gp0 = g[4 * N_L]; }
                }
                if (q == NI && copy_last) { z = gz0; geom = gg0; pq = gp0; }
                const double zi = 1.0 / z;
                const bool vis = geom != 0.0 && pq >= -1.0;
                KN[q].ph = x;
                KN[q].live = vis ? 1 : 0;
                if (ATM == 1) {
                    KN[q].x = zi * (TUnit<R>::v / kT);
                    KN[q].g = vis ? (R)(geom * (zi * zi * zi)) : (R)0;
                }
                if (q < NI) {
                    const double wd = xn - x;
                    KN[q].h = (R)wd;
                    KN[q].ih = (R)(1.0 / wd);
                }
            }
            if (I == 0) {
                // the parallel's cells: azimuths and their order, the largest area
                double amax = 0.0;
                int bad = 0;                            // bit 0: not one increasing turn, bit 1: not evenly spaced
                for (int j = tid; j < S; j += NT) {
                    if (j != tid) {
                        ca = area[j];
                        cr = radp ? radp[j] == 1 : ca > 0.0;
                        cp = prow[j];
                        cp1 = prow[min(j + 1, S - 1)];
                    }
                    CELL[j].phi = cp;
                    const double d = (cp_last - cp_first) / (double)(S - 1);
                    if (j + 1 < S ? !(cp1 > cp) : !(cp - cp_first < TWO_PI)) bad |= 1;
                    // evenly spaced to rounding
                    if (!(fabs(cp - (cp_first + (double)j * d)) <= 8.0 * DBL_EPSILON * (fabs(cp_first) + fabs(cp_last)))) bad |= 2;
                    if (cr && ca > 0.0) amax = fmax(amax, ca);
                }
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) amax = fmax(amax, __shfl_xor(amax, o, 64));
                const bool b1 = __ballot(bad & 1) != 0ull, b2 = __ballot(bad & 2) != 0ull;
                if (lane == 0) { AM[w] = amax; AF[w] = (b1 ? 1 : 0) | (b2 ? 2 : 0); }
            }
            __syncthreads();
            const double lo = KN[0].ph, hi = KN[NI].ph;
            if (I == 0) {
                double amax = 0.0;
                int bad = 0;
#pragma unroll
                for (int q = 0; q < NW; q++) { amax = fmax(amax, AM[q]); bad |= AF[q]; }
                order = (bad & 1) ? 0 : (bad ? 1 : 2);
                a_ref = sizeof(R) == 4 && amax > 0.0 ? amax : 1.0;
                invd = (double)(S - 1) / (CELL[S - 1].phi - CELL[0].phi);
                for (int j = tid; j < S; j += NT) {
                    if (j != tid || S > NT) {
                        ca = area[j];
                        cr = radp ? radp[j] == 1 : ca > 0.0;
                    }
                    CELL[j].area = cr ? (R)(sizeof(R) == 4 ? ca / a_ref : ca) : (R)__builtin_nan("");
                    // how far the like cells go from here (full ones, dark ones; within
                    // 64): evenly spaced, their moments have a closed form
                    const unsigned long long mf = __ballot(cr && ca == amax), mz = __ballot(!cr);
                    const unsigned long long like = ((cr && ca == amax) ? mf : (cr ? 0ull : mz)) >> lane;
                    const int len = __ffsll((long long)~like);
                    CELL[j].run = order == 2 && like ? (len ? len - 1 : 64) : 1;
                }
            }
            // pieces whose Akima stencil (secants i-2 .. i+2, periodic) shows a leaf
            for (int q = tid; q < NI; q += NT) {
                int any = 0;
#pragma unroll
                for (int d = -2; d <= 3; d++) {
                    int k = q + d;
                    k = k < 0 ? k + NI : (k > NI ? k - NI : k);
                    any |= KN[k].live;
                }
                KN[q].stencil = any;
            }
            if (w == NW - 1) {
                // a phase's turn of the cells: the first cell after the wrap, and
                // the first point and the wrap's shift of the cells from there on
                // (a) and of those before it (b)
                SlabPhase t{0.0, 0.0, 0.0, 0.0, 0, 0};
                if (np > 0 && order > 0) {
                    const double x0 = wrap_phase(php + CELL[0].phi, lo, hi);
                    int a = 1, b = S;
                    while (a < b) {
                        const int mid = (a + b) >> 1;
                        if (wrap_phase(php + CELL[mid].phi, lo, hi) < x0) b = mid;
                        else a = mid + 1;
                    }
                    t.j0 = a == S ? 0 : a;
                    const double sa = php + CELL[t.j0].phi;
                    t.xa = wrap_phase(sa, lo, hi);
                    t.oa = t.xa - sa;
                    if (t.j0 > 0) { t.xb = x0; t.ob = x0 - (php + CELL[0].phi); }
                }
                PL[lane] = t;
            }
            // the pieces of this wavefront's quarter: a window that slides from
            // interval to interval (lanes = energies), kept in registers
            const int q_end = min((rq + 1) * Q, NI);
            R y0 = (R)0, y1 = (R)0, y2 = (R)0;          // profile at knots i, i + 1, i + 2
            R sm1 = (R)0, s0 = (R)0, s1 = (R)0;         // secants of intervals i - 1, i, i + 1
            R d0 = (R)0, d1 = (R)0;                     // |s0 - sm1|, |s1 - s0|
            R tl = (R)0;                                // slope at knot i
            bool flat = true;                           // that knot's weights are zero
            auto knot = [&](int k) -> R {               // k from -2 to NI + 2 over the periodic turn
                const int q = k < 0 ? k + NI : (k > NI ? k - NI : k);
                R y = (R)0;
                if (KN[q].live) {                       // the same for the whole wavefront
                    if (ATM == 1) {
                        const double t = E * KN[q].x;
                        R f = planck_factor(t, (R)0);
                        if (correct) f -= planck_factor(t * x_else, (R)0);
                        y = f * KN[q].g;
                    } else y = prof[(size_t)(q == NI ? 0 : q) * N_E];
                }
                return e_ok ? y : (R)0;
            };
            // The window is formed afresh where a block's slabs begin and slid from there,
            // and how many blocks share a parallel depends on the batch: both ways round
            // alike (no product of one fused into another's sum by the compiler's
            // choice), so a request's FP32 pieces are the same in any batch.
            auto secant = [&](R ya, R yb, int k) -> R {  // of interval k
#pragma clang fp contract(off)
                return (yb - ya) * KN[k < 0 ? k + NI : (k >= NI ? k - NI : k)].ih;
            };
            // slope at a knot from the secants a, b before and c, d after it (|b - a| = wl, |d - c| = wr)
            auto slope = [&](R b, R c, R wl, R wr, bool& fl) -> R {
                const R ws = wl + wr;
                fl = sizeof(R) == 4 ? ws < (R)FLT_MIN : ws == (R)0;   // quot needs a normal divisor
                const R al = fl ? (R)0 : quot(wl, ws);
                {
#pragma clang fp contract(off)
                    const R rest = ((R)1 - al) * b;
                    return fma(al, c, rest);
                }
            };
            unsigned live = 0u;
            // s_begin - 1: the first slab's operands alone
#pragma unroll 1
            for (int s = s_begin - 1; s < s_end; s++) {
                __syncthreads();
                const int buf = (s + 1) & 1, nb = buf;  // slab s + 1 goes to buffer (s + 1) & 1, slab s is in the other
                const int pb = buf ^ 1;
                const unsigned live_s = live;
                live = 0u;
                if (s + 1 < s_end) {
                    const int lq = lane / RUN, iv = lq * Q + (s + 1) * RUN + lane % RUN;
                    live = (unsigned)__ballot(lane < SL && iv < min((lq + 1) * Q, NI) && KN[min(iv, NI)].stencil);
                }
                auto produce = [&]() {
                    if (s + 1 >= s_end) return;
                    const int ia = rq * Q + (s + 1) * RUN;
                    if (chunk_on && ia < q_end) {
                        const int lane = fresh(tid & 63);
                        if (s < s_begin) {              // the window's start
                            const R ym2 = knot(ia - 2), ym1 = knot(ia - 1);
                            y0 = knot(ia);
                            y1 = knot(ia + 1);
                            y2 = knot(ia + 2);
                            const R sm2 = secant(ym2, ym1, ia - 2);
                            sm1 = secant(ym1, y0, ia - 1);
                            s0 = secant(y0, y1, ia);
                            s1 = secant(y1, y2, ia + 1);
                            d0 = fabs(s0 - sm1);
                            d1 = fabs(s1 - s0);
                            tl = slope(sm1, s0, fabs(sm1 - sm2), d1, flat);
                        }
                        R* co = CO + ((size_t)(nb * SL + rq * RUN) * EC + ec) * 256 + (lane & 15) * 4 + (lane >> 4);
#pragma unroll
                        for (int k = 0; k < RUN; k++) {
                            const int iv = ia + k;
                            if (iv >= q_end) break;
                            const R y3 = knot(iv + 3), s2 = secant(y2, y3, iv + 2), d2 = fabs(s2 - s1);
                            bool flat1;
                            const R tr = slope(s0, s1, d0, d2, flat1);
                            if ((live >> (rq * RUN + k)) & 1u) {
                                const R h = KN[iv].h, ih = KN[iv].ih;
                                R b = s0, c = (R)0, d = (R)0;
                                const R te = flat1 ? s0 : tr;
                                if (!flat) {
                                    b = tl;
                                    c = ((R)3 * s0 - (R)2 * b - te) * ih;
                                    d = (b + te - (R)2 * s0) * (ih * ih);
                                }
                                // the Bernstein points bound the piece; where they leave its
                                // sign open its extremes settle it
                                const R h3 = h * (R)(1.0 / 3.0), b1 = y0 + b * h3, b2 = y1 - te * h3;
                                const R blo = fmin(fmin(y0, y1), fmin(b1, b2)), bhi = fmax(fmax(y0, y1), fmax(b1, b2));
                                int cls = (blo != (R)0 || bhi != (R)0) ? 1 : 0;
                                if (!correct && blo < (R)0) cls = open_class<R>(y0, b, c, d, h);
                                const bool on = cls != 0;
                                R* ck = co + (size_t)k * EC * 256;
                                ck[0] = on ? y0 : (R)0;
                                ck[64] = on ? b : (R)0;
                                ck[128] = on ? c : (R)0;
                                ck[192] = on ? d : (R)0;
                                const unsigned long long mt = __ballot(cls == 1), mx = __ballot(cls == 2);
                                if (lane == 0) {
                                    const int o = (nb * SL + rq * RUN + k) * EC + ec;
                                    ANZ[o] = mt;
                                    MIXM[o] = mx;
                                }
                            }
                            // the window moves on
                            y0 = y1; y1 = y2; y2 = y3;
                            sm1 = s0; s0 = s1; s1 = s2;
                            d0 = d1; d1 = d2;
                            tl = tr;
                            flat = flat1;
                        }
                    }
                    // moments (lanes = phases)
                    const int ma = w * MRUN;
                    if (ma < SL && ((live >> ma) & ((1u << MRUN) - 1u))) {
                        const int lane = fresh(tid & 63);
                        const SlabPhase t = PL[lane];
                        // cells (in turn order) whose point lies below b
                        auto below = [&](double b) -> int {
                            if (order == 2) {
                                // evenly spaced: a cell whose point rounds across b counts
                                // on either side, where the spline is continuous
                                const double fa = ceil((b - t.xa) * invd), fb = ceil((b - t.xb) * invd);
                                const int na = np - min(t.j0, np), nb2 = np - na;
                                return (int)fmin(fmax(fa, 0.0), (double)na) + (int)fmin(fmax(fb, 0.0), (double)nb2);
                            }
                            int a = 0, c = np;
                            while (a < c) {
                                const int mid = (a + c) >> 1;
                                int j = t.j0 + mid;
                                j = j >= S ? j - S : j;
                                if (wrap_phase(php + CELL[j].phi, lo, hi) < b) a = mid + 1;
                                else c = mid;
                            }
                            return a;
                        };
                        const R dsp = (R)(1.0 / invd);
                        const int ib = (ma / RUN) * Q + (s + 1) * RUN + ma % RUN;
                        int cur = order && ib > 0 ? below(KN[ib].ph) : 0;
#pragma unroll 1
                        for (int k = 0; k < MRUN; k++) {
                            const int iv = ib + k, o = nb * SL + ma + k;
                            if (iv >= NI) break;
                            const double lb = KN[iv].ph, ub = iv < NI - 1 ? KN[iv + 1].ph : __builtin_inf();
                            R M0 = (R)0, M1 = (R)0, M2 = (R)0, M3 = (R)0;
                            bool any = false;
                            const int first = cur;
                            // n cells of area ar at x, x + d, ..
                            auto add = [&](double x, R ar, int n) {
                                if (isnan(ar)) return;
                                const R t = (R)(x - lb), q = (R)n, q1 = (R)(n - 1);
                                const R k1 = dsp * ((R)0.5 * q * q1), k2 = dsp * dsp * (q * q1 * (R)(2 * n - 1) * (R)(1.0 / 6.0));
                                const R k3 = dsp * (k1 * k1);   // sums of k d, (k d)^2, (k d)^3
                                M0 += ar * q;
                                M1 += ar * (q * t + k1);
                                M2 += ar * ((q * t + (R)2 * k1) * t + k2);
                                M3 += ar * (((q * t + (R)3 * k1) * t + (R)3 * k2) * t + k3);
                                any = true;
                            };
                            if (order) {
                                const int nxt = iv < NI - 1 ? below(ub) : np;
                                while (cur < nxt) {
                                    int j = t.j0 + cur;
                                    const bool second = j >= S;
                                    j = second ? j - S : j;
                                    const SlabCell<R> cl = CELL[j];
                                    const int n = min(cl.run, nxt - cur);
                                    add((php + cl.phi) + (second ? t.ob : t.oa), cl.area, n);
                                    cur += n;
                                }
                            } else {
                                for (int j = 0; j < np; j++) {
                                    const double x = wrap_phase(php + CELL[j].phi, lo, hi);
                                    if (x < ub && (iv == 0 || x >= lb)) add(x, CELL[j].area, 1);
                                }
                            }
                            R* mo = MOM + o * 256 + (lane >> 4) * 64 + (lane & 15);
                            mo[0] = M0; mo[16] = M1; mo[32] = M2; mo[48] = M3;
                            CF[o * 64 + lane] = first | ((cur - first) << 16);
                            const unsigned long long nz = __ballot(any);
                            if (lane == 0) MASK[o] = nz;
                        }
                    }
                };
                auto products = [&]() {
                    if (!tile_on || !live_s) return;
                    const int lane = fresh(tid & 63);
                    bool hit = false, mixed = false;
                    if (lane < SL && ((live_s >> lane) & 1u) && ((MASK[pb * SL + lane] >> (16 * rq)) & 0xffffull)) {
                        hit = ANZ[(pb * SL + lane) * EC + ec] != 0ull;
                        mixed = MIXM[(pb * SL + lane) * EC + ec] != 0ull;
                    }
                    const unsigned mf = (unsigned)__ballot(hit);
                    unsigned mx = (unsigned)__ballot(mixed);
                    const unsigned mxa = mx;
                    const R* ca = CO + ((size_t)pb * SL * EC + ec) * 256 + 4 * lane;
                    const R* mb = MOM + pb * SL * 256 + rq * 64 + lane;
                    // NC tiles from tile c0 on; the next interval's operands are read while
                    // this one's products run
                    constexpr int NC = sizeof(R) == 4 ? 2 : 4;
#pragma unroll
                    for (int c0 = 0; c0 < 4; c0 += NC) {
                        R a[NC], an[NC], b = (R)0, bn = (R)0;
                        auto fetch = [&](int iv, R (&x)[NC], R& y) {
#pragma unroll
                            for (int c = 0; c < NC; c++) x[c] = ca[(size_t)iv * EC * 256 + c0 + c];
                            y = mb[iv * 256];
                            if ((mxa >> iv) & 1u) {         // sign-changing pieces stay out of the products
                                const unsigned long long mm = MIXM[(pb * SL + iv) * EC + ec] >> (lane & 15);
#pragma unroll
                                for (int c = 0; c < NC; c++)
                                    if ((mm >> (16 * (c0 + c))) & 1ull) x[c] = (R)0;
                            }
                        };
                        unsigned m = mf;
                        typename Mfma<R>::v4 sum[NC];
#pragma unroll
                        for (int c = 0; c < NC; c++) {
                            if constexpr (sizeof(R) == 4) sum[c] = {0.f, 0.f, 0.f, 0.f};
                            else sum[c] = acc[c0 + c];
                        }
                        if (m) {
                            fetch(__builtin_ctz(m), a, b);
#pragma unroll 1
                            while (true) {
                                m &= m - 1u;
                                if (m) fetch(__builtin_ctz(m), an, bn);
#pragma unroll
                                for (int c = 0; c < NC; c++) sum[c] = Mfma<R>::step(a[c], b, sum[c]);
                                if (!m) break;
#pragma unroll
                                for (int c = 0; c < NC; c++) a[c] = an[c];
                                b = bn;
                            }
                        }
#pragma unroll
                        for (int c = 0; c < NC; c++) {
                            if constexpr (sizeof(R) == 4) {
#pragma unroll
                                for (int r = 0; r < 4; r++) acc[c0 + c][r] = fma((double)sum[c][r], a_ref, acc[c0 + c][r]);
                            } else acc[c0 + c] = sum[c];
                        }
                    }
                    // sign-changing pieces: the k-th cell of each of the tile's phases in
                    // the interval, its powers against the pieces' coefficients by
                    // the same product, clipped
                    const int jc = mx ? PL[16 * rq + (lane & 15)].j0 : 0;
                    const int er = lane & 15, pw = lane >> 4;
                    while (mx) {
                        const int sl = __builtin_ctz(mx);
                        mx &= mx - 1u;
                        const int iv = (sl / RUN) * Q + s * RUN + sl % RUN, o = pb * SL + sl;
                        const unsigned long long mm = MIXM[o * EC + ec] >> er;
                        const R* cr = CO + ((size_t)o * EC + ec) * 256 + 64 * pw + 4 * er;
                        typename Mfma<R>::v4 sum[4], z4 = {(R)0, (R)0, (R)0, (R)0};
                        R a[4];
#pragma unroll
                        for (int c = 0; c < 4; c++) {
                            a[c] = ((mm >> (16 * c)) & 1ull) ? cr[c] : (R)0;
                            sum[c] = z4;
                        }
                        const int f = CF[o * 64 + 16 * rq + (lane & 15)];
                        const int kb = order ? (f >> 16) : (pc < N_P ? S : 0), jb = order ? jc + (f & 0xffff) : 0;
                        const double lb = KN[iv].ph, ub = iv < NI - 1 ? KN[iv + 1].ph : __builtin_inf();
#pragma unroll 1
                        for (int k = 0; __ballot(k < kb); k++) {
                            R ar = (R)0, t = (R)0;
                            if (k < kb) {
                                int j = jb + k;
                                j = j >= S ? j - S : j;
                                const double x = wrap_phase(phc + CELL[j].phi, lo, hi);
                                const R aj = CELL[j].area;
                                if (!isnan(aj) && (order || (x < ub && (iv == 0 || x >= lb)))) {
                                    ar = aj;
                                    t = (R)(x - lb);
                                }
                            }
                            const R t2 = t * t, tp = pw == 0 ? (R)1 : (pw == 1 ? t : (pw == 2 ? t2 : t2 * t));
#pragma unroll
                            for (int c = 0; c < 4; c++) {
                                const typename Mfma<R>::v4 v = Mfma<R>::step(a[c], tp, z4);
#pragma unroll
                                for (int r = 0; r < 4; r++) {
                                    if constexpr (sizeof(R) == 4) sum[c][r] += ar * fmaxf(v[r], 0.f);
                                    else acc[c][r] += ar * fmax(v[r], 0.0);
                                }
                            }
                        }
                        if constexpr (sizeof(R) == 4)
#pragma unroll
                            for (int c = 0; c < 4; c++)
#pragma unroll
                                for (int r = 0; r < 4; r++) acc[c][r] += (double)sum[c][r] * a_ref;
                    }
                };
                // one half of the wavefronts starts with the next slab's operands, the
                // other with this slab's products, so both units are fed
#pragma unroll 1
                for (int h = 0; h < 2; h++) {
                    if ((w + h) & 1) produce();
                    else products();
                }
            }
            asm volatile("" ::"v"(touch));
        }
    }
    if (!tile_on) return;
    // the wavefront's sums into the flux: E^3 and the norms in FP64
    const double scale = ATM == 1 ? E * E * (BB_NORM / KEV / (sizeof(R) == 4 ? PROFILE_UNIT : 1.0))
                                  : 1.0 / (E * KEV * (sizeof(R) == 4 ? TABLE_UNIT : 1.0));
    double* flux = F.flux + (size_t)mi * N_E * N_P;
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int src = 16 * c + Mfma<R>::row(lane, r), ee = e0 + 64 * ec + src;
            const double v = acc[c][r];
            const double sc = __shfl(scale, src, 64);
            if (ee < N_E && pc < N_P && v != 0.0) unsafeAtomicAdd(flux + (size_t)ee * N_P + pc, v * sc);
        }
}

// The table atmosphere's profiles, formed once per parallel and image for every
// energy (the fold's blocks of one parallel, two to eight of them, would each form their own).
//
// k_table_items numbers the contributing (parallel, image) pairs of the launch:
// item0[member][parallel] is the parallel's first, *total their count.
__global__ void __launch_bounds__(256) k_table_items(const Member* __restrict__ members, Layout L,
                                                     const int* __restrict__ valid, int* __restrict__ item0,
                                                     int* __restrict__ total)
{
    const int mi = blockIdx.x, tid = threadIdx.x;
    const Member& m = members[mi];
    if (!m.active || m.status) return;
    __shared__ int n_s, base_s;
    if (tid == 0) n_s = 0;
    __syncthreads();
    for (int i0 = 0; i0 < m.S; i0 += 256) {
        const int i = i0 + tid;
        int n = 0;
        if (i < m.S)
            while (n < L.IO_max && valid[((size_t)mi * L.S_max + i) * L.IO_max + n]) n++;
        // places within the member by an LDS counter: any order will do
        if (i < m.S) item0[(size_t)mi * L.S_max + i] = n ? atomicAdd(&n_s, n) : -1;
    }
    __syncthreads();
    if (tid == 0) base_s = atomicAdd(total, n_s);
    __syncthreads();
    for (int i = tid; i < m.S; i += 256) {
        int* p = item0 + (size_t)mi * L.S_max + i;
        *p = *p < 0 ? INT_MIN : *p + base_s;
    }
}

// k_table_profile: block per (parallel, member) of the pass, its images in turn.
// Four visible leaves at a time, the parallel's contracted table (k_table_slab)
// is contracted over the leaf's four mu nodes into LDS rows over the energy axis,
// read by consecutive threads; then a thread per energy takes its four nodes
// from the row: four LDS reads a value in place of sixteen gathered ones, and
// the values of 256 energies go out as one row.  A leaf's first energy
// follows another leaf's (or parallel's) last query, so it takes the
// reference's base-node history in full (num4d_I).
template <typename R>
__global__ void __launch_bounds__(256) k_table_profile(const Member* __restrict__ members, Layout L, FoldArgs F)
{
    const int i = blockIdx.x, mi = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const Member& m = members[mi];
    if (!m.active || m.status || i >= m.S || *F.item_total <= F.pass * F.cap) return;
    const size_t ro = (size_t)mi * L.S_max + i;
    const long long slot = (long long)F.item0[ro] - (long long)F.pass * F.cap;
    if (slot < 0 || slot >= F.cap) return;
    const int N_L = L.N_L, N_E = L.N_E, NI = N_L - 1, N2 = F.atm_N[2], N3 = F.atm_N[3];
    extern __shared__ __align__(16) double tsm[];
    double* X3 = tsm;                     // [N3] energy axis
    double* S3 = X3 + N3;                 // [4 (N3 - 3)] its Lagrange denominators
    double* ROW = S3 + 4 * (N3 - 3);      // [2][4][N3] two sets of four rows
    TableKnot* KT = (TableKnot*)(ROW + 8 * N3);   // [N_L]
    int* LIST = (int*)(KT + N_L);         // [N_L] visible leaves
    __shared__ int n_live;
    const double* x2 = F.atm_axes + F.atm_N[0] + F.atm_N[1];
    const double* S2 = F.atm_S + 4 * ((F.atm_N[0] - 3) + (F.atm_N[1] - 3));
    for (int q = tid; q < N3; q += 256) X3[q] = x2[N2 + q];
    for (int q = tid; q < 4 * (N3 - 3); q += 256) S3[q] = S2[4 * (N2 - 3) + q];
    const double* slab = F.slab + ro * (size_t)N2 * N3;
    const double kT = K_B_OVER_KEV * pow(10.0, F.logT[ro]), lkT = log10(kT);
    const double norm = pow(10.0, 3.0 * F.logT[ro]) * NUM4D_NORM;
    const double kT_else = K_B_OVER_KEV * pow(10.0, m.else_logT);
    const double unit = sizeof(R) == 4 ? TABLE_UNIT : 1.0;
    for (int I = 0; I < L.IO_max; I++) {
        const size_t vix = ro * L.IO_max + I;
        if (!F.valid[vix]) break;
        const double* g = F.geo + vix * 5 * N_L;
        __syncthreads();                  // the previous image's reads are done
        if (tid == 0) n_live = 0;
        __syncthreads();
        for (int q = tid; q < N_L; q += 256) {
            const double geom = g[3 * N_L + q], pq = g[4 * N_L + q], zi = 1.0 / g[N_L + q], mu = g[2 * N_L + q];
            if (!(geom != 0.0 && pq >= -1.0)) continue;
            TableKnot& k = KT[q];
            k.lq = log10(zi) - lkT;
            k.zi = zi;
            k.geom = geom * unit;
            k.b = n4_base(x2, N2, mu);
            n4_weights_pre(x2, k.b, mu, S2 + 4 * k.b, k.w);
            double vec[4], prev[4], st[5];
            int has_prev = 1;
            const int kd = (int)pq;
            vec[0] = F.logT[ro]; vec[1] = F.logg[ro]; vec[2] = mu;
            vec[3] = log10((F.energies[0] * zi) / kT);
            if (kd >= 0) {
                prev[0] = vec[0]; prev[1] = vec[1]; prev[2] = g[2 * N_L + kd];
                prev[3] = log10((F.energies[N_E - 1] / g[N_L + kd]) / kT);
            } else {
                prev_query_state(F, L, mi, i, I, st);
                if (st[0] > 0.5) { prev[0] = st[1]; prev[1] = st[2]; prev[2] = st[3]; prev[3] = st[4]; }
                else has_prev = 0;
            }
            k.y0 = num4d_I(F, vec, prev, has_prev) * NUM4D_NORM;
            LIST[atomicAdd(&n_live, 1)] = q;
        }
        __syncthreads();
        const int nl = n_live;
        R* out = (R*)F.prof + (size_t)(slot + I) * N_L * N_E;
        for (int n0 = 0; n0 < nl; n0 += 4) {
            double* row = ROW + ((n0 >> 2) & 1) * 4 * N3;
            const int nk = min(4, nl - n0);
            for (int q = tid; q < nk * N3; q += 256) {
                const int kk = q / N3, l = q - kk * N3;
                const TableKnot& k = KT[LIST[n0 + kk]];
                const double* r = slab + (size_t)k.b * N3 + l;
                row[q] = k.w[0] * r[0] + k.w[1] * r[N3] + k.w[2] * r[2 * (size_t)N3] + k.w[3] * r[3 * (size_t)N3];
            }
            __syncthreads();              // (the set before last is read no more)
            for (int e = tid; e < N_E; e += 256) {
                const double lE = F.logE[e], lEp = e > 0 ? F.logE[e - 1] : 0.0, E = F.energies[e];
                for (int kk = 0; kk < nk; kk++) {
                    const int q = LIST[n0 + kk];
                    const TableKnot& k = KT[q];
                    double In = k.y0;
                    if (e > 0) {
                        double v = lE + k.lq;
                        const double vp = lEp + k.lq;
                        int b;
                        // the energy axis clamps as the reference's base-node rule does
                        if (v > X3[N3 - 1]) {
                            b = N3 - 4;
                            if (vp < X3[N3 - 3]) v = X3[N3 - 1];
                        } else if (v < X3[0]) {
                            b = 0;
                            if (vp >= X3[2]) v = X3[0];
                        } else b = n4_base_near(X3, N3, v);
                        double w3[4];
                        n4_weights_pre(X3, b, v, S3 + 4 * b, w3);
                        const double* r = row + kk * N3 + b;
                        In = w3[0] * r[0] + w3[1] * r[1] + w3[2] * r[2] + w3[3] * r[3];
                        In = In < 0.0 ? 0.0 : In * norm;
                    }
                    if (m.correct) {
                        const double Ep = E * k.zi;
                        In -= Ep * Ep * Ep / (exp(Ep / kT_else) - 1.0) * BB_NORM;
                    }
                    out[(size_t)q * N_E + e] = (R)(In * k.geom);
                }
            }
        }
    }
}

template __global__ void k_table_profile<float>(const Member*, Layout, FoldArgs);
template __global__ void k_table_profile<double>(const Member*, Layout, FoldArgs);

template __global__ void k_slab_fold<float, 1, 1>(const Member*, Layout, FoldArgs);
template __global__ void k_slab_fold<float, 1, 2>(const Member*, Layout, FoldArgs);
template __global__ void k_slab_fold<float, 2, 1>(const Member*, Layout, FoldArgs);
template __global__ void k_slab_fold<float, 2, 2>(const Member*, Layout, FoldArgs);
template __global__ void k_slab_fold<double, 1, 1>(const Member*, Layout, FoldArgs);
template __global__ void k_slab_fold<double, 1, 2>(const Member*, Layout, FoldArgs);
template __global__ void k_slab_fold<double, 2, 2>(const Member*, Layout, FoldArgs);
template __global__ void k_slab_fold<double, 2, 1>(const Member*, Layout, FoldArgs);

}  // namespace xh
