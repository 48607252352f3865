// Henon-step glue around the hot path (src/cmc/cmc.c:240-407 order):
// energy_conservation1/2 (src/cmc/cmc_utils.c:2153-2227), tidally_strip_stars
// (src/cmc/cmc_evolution_thr.c:443-646, TIDAL_TREATMENT 0), ComputeIntermediateEnergy
// (cmc_utils.c:368-391), set_velocities3 (:254-354) and ComputeEnergy (:604-653).
// All are per-star streaming maps plus deterministic two-level reductions.
#include "kernels.hpp"

namespace {
constexpr int GT = 256;
__device__ __forceinline__ double sqr(double x) { return x * x; }

// Sums over GT threads by halving (off = GT / 2 .. 1: thread t < off adds thread t + off's), in
// v of thread 0: the first two halvings through LDS, the rest by shuffles of the first wave (one
// barrier, not nine).  t: the thread's index among the GT.
template <int NV>
__device__ __forceinline__ void tree_sum(double (&v)[NV], double (*lds)[GT], int t)
{
    static_assert(GT == 256, "two halvings down to a wave");
    for (int i = 0; i < NV; i++) lds[i][t] = v[i];
    __syncthreads();
    if (t < 64) {
        for (int i = 0; i < NV; i++) v[i] = (lds[i][t] + lds[i][t + 128]) + (lds[i][t + 64] + lds[i][t + 192]);
        for (int off = 32; off > 0; off >>= 1)
            for (int i = 0; i < NV; i++) v[i] += __shfl_down(v[i], off, 64);
    }
}

template <int NV>
__device__ void block_sum_store(double (&v)[NV], double *__restrict__ out)
{
    __shared__ double lds[NV][GT];
    tree_sum<NV>(v, lds, threadIdx.x);
    if (threadIdx.x == 0)
        for (int i = 0; i < NV; i++) out[i] = v[i];
}

// the sum of block partials, in res of thread 0
template <int NV>
__device__ void final_sum(const double *__restrict__ partials, int64_t nblocks, double (&res)[NV])
{
    __shared__ double lds[NV][GT];
    for (int i = 0; i < NV; i++) res[i] = 0.0;
#pragma unroll 8
    for (int64_t b = threadIdx.x; b < nblocks; b += GT)      // unrolled: independent loads in flight
        for (int i = 0; i < NV; i++) res[i] += partials[8 * b + i];
    tree_sum<NV>(res, lds, threadIdx.x);
}

struct ec1_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P)
{
    int64_t i = 1 + (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (i > s->n_max) return;
    double ri = f.r[i];
    f.vtold[i] = f.vt[i];
    f.vrold[i] = f.vr[i];
    f.Uoldrold[i] = f.phi[i] + phi_s_own(ri, f.m[i], P.inv_nstar, ri);
}
};

// energy_conservation2: Uoldrnew = potential(rnew) + MPI_PHI_S(rnew, i).  The orbit
// phase already evaluated potential(rnew) for sampled stars (flag 256) on the same
// arrays, so only circular / removed stars search here.
struct ec2_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P)
{
    int64_t i = 1 + (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    int64_t n = s->n_max;
    if (i > n) return;
    double x = f.rnew[i];
    double pot;
    int fl = f.flags[i];
    if (fl & 256) {
        pot = f.pot_rnew[i];
    } else {
        bool bad = false;
        pot = potential_at(f.r, f.phi, n, x, 1, n + 1, &bad);
        if (bad) dev_set_error(s, CMCG_E_BRACKET, i);
        f.pot_rnew[i] = pot;
        f.flags[i] = fl | 256;
    }
    f.Uoldrnew[i] = pot + phi_s_own(f.r[i], f.m[i], P.inv_nstar, x);
}
};

// The step's form of energy_conservation2 followed by ComputeIntermediateEnergy's
// first loop (cmc_utils.c:335-351): the stripping between them leaves every field
// that EI reads unchanged for the stars it keeps and sets EI = 0 for the stars it
// strips, so EI can be formed here, before it, with the same result.
// It also forms D = vold^2 + 2 (1 - q) (Uoldrold - Uoldrnew), the part of
// set_velocities3's vnew^2 (cmc_utils.c:242-247) that reaches it through the permutation
// in place of its four inputs: the same operations in the same order, so the same double.
// With strip_done it also begins the stripping loop that follows, and leaves every block's
// largest r_apo of the stars that loop may strip: a pass then reads the stars of the blocks
// that reach beyond the tidal radius only (16 -> 6 us at N = 4e6, 20 -> 3 in one block at 6e4).
struct ec2_ie_kernel {
    static constexpr int LB = GT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P, double *__restrict__ dpre,
                                               int32_t *strip_done, double *__restrict__ apo_max)
{
    __shared__ double wmax[GT / 64];
    const int64_t i = 1 + (int64_t)kg_.bid * GT + threadIdx.x;
    const int64_t n = s->n_max;
    if (i == 1 && strip_done) {
        s->Etidal = 0.0;        // cmc_evolution_thr.c:449
        *strip_done = 0;
    }
    double apo = 0.0;
    if (i <= n) {
        const double x = f.rnew[i];
        double pot;
        const int fl = f.flags[i];
        if (fl & 256) {
            pot = f.pot_rnew[i];
        } else {
            bool bad = false;
            pot = potential_at(f.r, f.phi, n, x, 1, n + 1, &bad);
            if (bad) dev_set_error(s, CMCG_E_BRACKET, i);
            f.pot_rnew[i] = pot;
            f.flags[i] = fl | 256;
        }
        const double Uoldrnew = pot + phi_s_own(f.r[i], f.m[i], P.inv_nstar, x);
        f.Uoldrnew[i] = Uoldrnew;
        if (x < 1.0e6) f.EI[i] = sqr(f.vr[i]) + sqr(f.vt[i]) + f.phi[i] - pot;
        const double q = 0.5;
        const double vtold = f.vtold[i], vrold = f.vrold[i];
        const double vold2 = vtold * vtold + vrold * vrold;
        dpre[i] = vold2 + 2.0 * (1.0 - q) * (f.Uoldrold[i] - Uoldrnew);
        if (apo_max && x < 1000000) apo = fmax(f.r_apo[i], 0.0);      // NaN: 0, beyond no radius, as in the pass
    }
    if (!apo_max) return;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const double other = __shfl_xor(apo, o, 64);
        apo = other > apo ? other : apo;
    }
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = apo;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < GT / 64; w++) apo = wmax[w] > apo ? wmax[w] : apo;
        apo_max[kg_.bid] = apo;
    }
}
};

struct strip_begin_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s, int32_t *done)
{
    s->Etidal = 0.0;        // cmc_evolution_thr.c:449
    *done = 0;
}
};

// One pass of the stripping loop (cmc_evolution_thr.c:447-645) is two kernels: a
// fixed grid in which every block derives Rtidal from the scalars left by the
// previous pass, strips its stars (grid-stride) and stores its partial sums, then one
// block that reduces them in block order, updates the scalars and decides whether the
// loop ends.  Passes after the end return at once, so a fixed number of passes can be
// enqueued (or captured in a graph) without a host round trip.
constexpr int STRIP_BLOCKS = 1024;
constexpr int STRIP_TAIL_PASSES = 64;     // after STRIP_GRAPH_PASSES grid passes of a captured step

// Star i in one pass: strip it if it is due and add its share to (Eescaped, Jescaped,
// DTidalMassLoss, Etidal).
__device__ __forceinline__ void strip_star(DevFields &f, const KParams &P, double Rt, int64_t n, int64_t i, double (&v)[4])
{
    if (i <= n && f.r_apo[i] > Rt && f.rnew[i] < 1000000) {
        double m = f.m[i], E = f.E[i], J = f.J[i];
        f.rnew[i] = CMCG_SF_INFINITY; f.vrnew[i] = 0.0; f.vtnew[i] = 0.0;
        f.knew[i] = -1;
        v[0] += E * m / (double)P.n_star;   // Eescaped
        v[1] += J * m / (double)P.n_star;   // Jescaped
        v[2] += m / (double)P.n_star;       // DTidalMassLoss
        v[3] += E * m / (double)P.n_star;   // Etidal
        // destroy_obj
        f.vr[i] = 0.0; f.vt[i] = 0.0; f.E[i] = 0.0; f.J[i] = 0.0; f.id[i] = 0;
        f.X[i] = 0.0; f.Y[i] = 0.0; f.r_peri[i] = 0.0; f.r_apo[i] = 0.0;
        f.rOld[i] = 0.0; f.Uoldrold[i] = 0.0; f.Uoldrnew[i] = 0.0; f.vrold[i] = 0.0; f.vtold[i] = 0.0;
        f.EI[i] = 0.0;
        f.m[i] = 2.2250738585072014e-308;
        f.flags[i] |= CMCG_SF_STRIPPED;
    }
}

// Block bi's share of one pass (stars 1 + bi*GT + t, stride nb*GT): strip them and
// store the block's partial sums.  apo_max (or null): bounds of r_apo per GT stars.
__device__ void strip_block(DevFields &f, const KParams &P, double Rt, int64_t n, double *__restrict__ partials,
                            unsigned nb, unsigned bi, const double *__restrict__ apo_max)
{
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int64_t b = bi; b * GT < n; b += nb)
        if (!apo_max || apo_max[b] > Rt) strip_star(f, P, Rt, n, 1 + b * GT + threadIdx.x, v);
    block_sum_store<4>(v, partials + 8 * bi);
}

__device__ __forceinline__ double strip_rtidal(const DevScalars *s, const KParams &P)
{
    return P.orbit_r * pow(s->Mtotal - (s->TidalMassLoss - s->OldTidalMassLoss), 1.0 / 3.0);
}

// The scalars at the end of a pass with sums res (one thread), and the loop's exit
__device__ void strip_update(DevScalars *s, double Rt, const double (&res)[4], int32_t *done)
{
    s->Rtidal = Rt;
    s->Eescaped += res[0];
    s->Jescaped += res[1];
    s->Etidal += res[3];
    s->TidalMassLoss += res[2];
    s->DTidalMassLoss = res[2];
    if (!(res[2] > 0)) *done = 1;
}

// The end of a pass: the block partials summed in block order, the scalars updated,
// the loop's exit decided (all threads of the calling block take part).
__device__ void strip_finish(DevScalars *s, double Rt, int32_t *done, const double *__restrict__ partials,
                             unsigned nb)
{
    double res[4];
    final_sum<4>(partials, nb, res);
    if (threadIdx.x == 0) strip_update(s, Rt, res, done);
}

struct strip_pass_kernel {
    static constexpr int LB = GT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P, const int32_t *done,
                                               double *__restrict__ partials, const double *__restrict__ apo_max)
    {
        if (*done) return;
        strip_block(f, P, strip_rtidal(s, P), s->n_max, partials, kg_.nb, kg_.bid, apo_max);
    }
};

struct strip_end_kernel {
    static constexpr int LB = GT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s, KParams P, int32_t *done,
                                               const double *__restrict__ partials, unsigned nb)
    {
        if (*done) return;
        strip_finish(s, strip_rtidal(s, P), done, partials, nb);
    }
};

// The rest of the loop in one block, for a captured step: after the grid passes the
// loop has nearly always ended and this returns at once; otherwise it runs further
// passes here, at most STRIP_TAIL_PASSES (then the step reports CMCG_E_STRIP).  The
// block plays the nb blocks of a grid pass one after another and writes the same
// partials, so the sums add in the same order as in the eager loop.
struct strip_tail_kernel {
    static constexpr int LB = GT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P, int32_t *done,
                                                        double *__restrict__ partials, unsigned nb,
                                                        const double *__restrict__ apo_max)
{
    __shared__ int32_t sdone;
    for (int pass = 0; pass < STRIP_TAIL_PASSES; pass++) {
        if (threadIdx.x == 0) sdone = *(volatile int32_t *)done;
        __syncthreads();
        if (sdone) return;
        const double Rt = strip_rtidal(s, P);
        const int64_t n = s->n_max;
        __syncthreads();
        for (unsigned bi = 0; bi < nb; bi++) {
            strip_block(f, P, Rt, n, partials, nb, bi, apo_max);
            __syncthreads();               // its LDS is reused
        }
        __threadfence_block();
        __syncthreads();
        strip_finish(s, Rt, done, partials, nb);
        __threadfence();
        __syncthreads();
    }
    if (threadIdx.x == 0 && !*(volatile int32_t *)done) dev_set_error(s, CMCG_E_STRIP, 0);
}
};

// The whole loop in one block for a cluster of at most STRIP_ONE stars: a pass strips and sums
// only the groups of four blocks of the grid pass that may have something to strip, by the 256
// threads that play each of their blocks with the same tree; the other blocks' sums are zero.
// So the sums are those of the grid passes.  (A pass and its end took 9 us in two launches,
// however few the stars, and a step has two passes at least, or in a captured step three and
// the tail, 31 us; here all passes take 6 us at 1e4 stars, 23 at 6e4 of a King cluster at its tidal
// radius.)
constexpr int64_t STRIP_ONE = 65536;
constexpr int STRIP_ONE_T = 1024;
struct strip_one_kernel {
    static constexpr int LB = STRIP_ONE_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P, int32_t *done,
                                               int max_passes, bool report, const double *__restrict__ apo_max)
{
    __shared__ double lds[4][4][GT];
    __shared__ double blk[4][STRIP_ONE / GT];      // the grid pass's block sums
    __shared__ uint32_t found[STRIP_ONE / STRIP_ONE_T];
    __shared__ bool more;
    const int t = threadIdx.x, vt = t & (GT - 1), sub = t >> 8;
    const int64_t n = s->n_max;
    const int groups = (int)((n + STRIP_ONE_T - 1) / STRIP_ONE_T);
    for (int pass = 0; pass < max_passes; pass++) {
        const double Rt = strip_rtidal(s, P);
        if (t < groups) {
            bool b = false;
            for (int q = 0; q < 4; q++) b |= (int64_t)(4 * t + q) * GT < n && apo_max[4 * t + q] > Rt;
            found[t] = b;
        }
        if (t < STRIP_ONE / GT)
            for (int q = 0; q < 4; q++) blk[q][t] = 0.0;
        __syncthreads();
        bool any = false;
        for (int g = 0; g < groups; g++) {
            if (!found[g]) continue;
            any = true;
            double v[4] = {0.0, 0.0, 0.0, 0.0};
            strip_star(f, P, Rt, n, 1 + (int64_t)g * STRIP_ONE_T + t, v);
            tree_sum<4>(v, lds[sub], vt);
            if (vt == 0)
                for (int q = 0; q < 4; q++) blk[q][4 * g + sub] = v[q];
            __syncthreads();
        }
        // final_sum over the grid pass's block sums: its thread b holds block b alone here
        double res[4] = {0.0, 0.0, 0.0, 0.0};
        if (any) {
            if (sub == 0)
                for (int q = 0; q < 4; q++) res[q] = blk[q][vt];
            tree_sum<4>(res, lds[sub], vt);
        }
        if (t == 0) {
            strip_update(s, Rt, res, done);
            more = res[2] > 0;
        }
        __threadfence_block();
        __syncthreads();
        if (!more) return;
    }
    if (t == 0 && report) dev_set_error(s, CMCG_E_STRIP, 0);
}
};

// ComputeIntermediateEnergy, first loop (EI).
struct ie_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s)
{
    int64_t j = 1 + (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    int64_t n = s->n_max;
    if (j > n) return;
    double x = f.rnew[j];
    if (x < 1.0e6) {
        double pot;
        if (f.flags[j] & 256) pot = f.pot_rnew[j];
        else {
            bool bad = false;
            pot = potential_at(f.r, f.phi, n, x, 1, n + 1, &bad);
            if (bad) dev_set_error(s, CMCG_E_BRACKET, j);
        }
        f.EI[j] = sqr(f.vr[j]) + sqr(f.vt[j]) + f.phi[j] - pot;
    }
}
};

// ComputeIntermediateEnergy, second loop (transfer of the new orbit variables).
struct ie_transfer_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s)
{
    int64_t j = 1 + (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (j > s->n_max) return;
    f.rOld[j] = f.r[j];
    f.r[j] = f.rnew[j];
    f.vr[j] = f.vrnew[j];
    f.vt[j] = f.vtnew[j];
}
};

// set_velocities3 per-star part.  Stars with vnew2 <= 0 ("events") carry excess
// energy that the following stars absorb (cmc_utils.c:268-310); they are counted
// per block for an ordered compaction.
// potential(r) of the new potential at every old node.  The old radii (the array the
// sort read, left intact in the alternate buffer) are sorted, so a block's MERGE_BLK
// consecutive old radii [x_first, x_last] fall into one contiguous run of new nodes:
// two waves find its ends, the block stages the run in LDS (coalesced)
// and every radius is placed by bisection in LDS.  A run longer than MERGE_LDS nodes
// is searched in global memory within the same ends.  The interval is the largest
// k with r_k < x, as in potential_at (the search predicate is monotone, so any bracket
// holding that k gives the same k), and the interpolation is the same expression, so
// the values equal potential_at(x) bit for bit.
constexpr int MERGE_T = 256, MERGE_PER = 2, MERGE_BLK = MERGE_T * MERGE_PER, MERGE_LDS = 1024;

// Largest k in [1, n + 1] with r_k < x (1 if none) by a whole wave: 64 probes split the range
// into 65, four rounds at N = 4e6 where a bisection takes 22.  Uniform over the wave.
__device__ __forceinline__ int64_t wave_find_zero_r(const PackedNodes &nd, int64_t n, double x)
{
    const int lane = threadIdx.x & 63;
    int64_t lo = 1, hi = n + 1;
    while (lo < hi) {
        const int64_t step = (hi - lo) / 65 + 1, p = lo + (lane + 1) * step;     // lo + 65 step > hi
        const int c = (int)__popcll(__ballot(p <= hi && nd.R(p) < x));
        const int64_t top = lo + (c + 1) * step - 1;
        lo += c * step;
        hi = top < hi ? top : hi;
    }
    return lo;
}

struct old_node_potential_kernel {
    static constexpr int LB = MERGE_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ r_old,
                                                                     const double2 *__restrict__ nodes,
                                                                     DevScalars *s, double2 *__restrict__ u_old,
                                                                     const double *__restrict__ dpre)
{
    __shared__ double2 L[MERGE_LDS];
    __shared__ int64_t ends[2];
    const int64_t n_old = s->sort_in, n = s->n_max;
    const int64_t first = 1 + (int64_t)kg_.bid * MERGE_BLK;
    if (first > n_old) return;
    const int64_t last = first + MERGE_BLK - 1 <= n_old ? first + MERGE_BLK - 1 : n_old;
    const PackedNodes nd{nodes};
    const double r1 = nd.R(1);
    const int t = threadIdx.x;
    const double xf = r_old[first], xl = r_old[last];
    if (t < 128) {                                 // wave 0: the first's, wave 1: the last's
        const double x = t < 64 ? xf : xl;
        const int64_t k = x == 0.0 || x < r1 ? 1 : wave_find_zero_r(nd, n, x);
        if ((t & 63) == 0) ends[t >> 6] = k;
    }
    __syncthreads();
    const int64_t lo = ends[0], hi = ends[1];
    const int64_t span = hi + 2 - lo;             // nodes lo .. hi+1
    const bool staged = span <= MERGE_LDS && hi + 1 <= n + 1;
    if (staged)
        for (int64_t k = t; k < span; k += MERGE_T) L[k] = nodes[lo + k];
    __syncthreads();
    for (int u = 0; u < MERGE_PER; u++) {
        const int64_t sl = first + t + (int64_t)u * MERGE_T;
        if (sl > last) break;
        const double x = r_old[sl];
        double v;
        if (x == 0.0 || x < r1 || !(x >= xf && x <= xl)) {    // the latter only if unsorted
            bool bad = false;
            v = potential_at_n(nd, n, x, 1, n + 1, &bad);
            if (bad) dev_set_error(s, CMCG_E_BRACKET, sl);
        } else {
            int64_t i;
            double ri, pi, ri1, pi1;
            if (staged) {
                int a = 0, b = (int)(hi - lo);
                while (a < b) {
                    const int m = (a + b + 1) >> 1;
                    if (L[m].x < x) a = m;
                    else b = m - 1;
                }
                i = lo + a;
                ri = L[a].x; pi = L[a].y; ri1 = L[a + 1].x; pi1 = L[a + 1].y;
            } else {
                i = lo == hi ? lo : find_zero_r_n(nd, lo, hi, x);
                nd.RP(i, ri, pi);
                if (i + 1 <= n + 1) nd.RP(i + 1, ri1, pi1);
                else { ri1 = ri; pi1 = pi; }
            }
            if (i > n) { dev_set_error(s, CMCG_E_BRACKET, sl); v = 0.0; }
            else v = pi + (pi1 - pi) * (1.0 / ri - 1.0 / x) / (1.0 / ri - 1.0 / ri1);
        }
        // with the radius and D in one 32-byte sector: set_velocities3 reads them at once
        u_old[2 * sl] = make_double2(v, x);
        u_old[2 * sl + 1] = make_double2(dpre[sl], 0.0);
    }
}
};

constexpr int SV3_COARSE = 1024;      // LDS samples of r for potential(rOld)

// With u_old (the step): potential(rOld), rOld itself and D (in place of vtold, vrold,
// Uoldrold and Uoldrnew) through the sort's permutation.  Without: the
// reference's fields and a search (the entry point of the reference's name).
struct sv3_kernel {
    static constexpr int LB = GT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P, double *__restrict__ excess_c,
                                                 int64_t *__restrict__ blk_cnt, const double2 *__restrict__ mid,
                                                 const double2 *__restrict__ nodes, const double2 *__restrict__ u_old,
                                                 const uint32_t *__restrict__ perm, int64_t *__restrict__ blk_events)
{
    __shared__ int wcnt[GT / 64];
    __shared__ double cr[SV3_COARSE + 1];
    bool event = false;
    const double q = 0.5;
    int64_t i = 1 + (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    int64_t n = s->n_max;
    Coarse C;
    C.cr = cr; C.cphi = nullptr; C.cs = SV3_COARSE; C.n1 = n + 1; C.hint = false;
    C.mid = mid;
    C.stride = coarse_stride(n, SV3_COARSE);
    if (!u_old)      // the samples serve only the search for potential(rOld)
        for (int sI = threadIdx.x; sI <= SV3_COARSE; sI += blockDim.x) cr[sI] = f.r[coarse_k(C, sI)];
    __syncthreads();
    if (i <= n) {
        double m = f.m[i], ri = f.r[i];
        double Unewrold, D;
        if (u_old) {
            const int64_t old = 2 * (int64_t)perm[i - 1];
            const double2 ux = u_old[old];
            D = u_old[old + 1].x;
            Unewrold = ux.x + phi_s_own(ri, m, P.inv_nstar, ux.y);
        } else {
            const double rO = f.rOld[i];
            bool bad = false;
            Unewrold = potential_at_coarse_n(PackedNodes{nodes}, n, rO, 1, n + 1, C, &bad) +
                       phi_s_own(ri, m, P.inv_nstar, rO);
            if (bad) dev_set_error(s, CMCG_E_BRACKET, i);
            const double vtold = f.vtold[i], vrold = f.vrold[i];
            const double vold2 = vtold * vtold + vrold * vrold;
            D = vold2 + 2.0 * (1.0 - q) * (f.Uoldrold[i] - f.Uoldrnew[i]);
        }
        double Unewrnew = f.phi[i] + phi_s_own(ri, m, P.inv_nstar, ri);
        double vnew2 = D + 2.0 * q * (Unewrold - Unewrnew);
        double vr = f.vr[i], vt = f.vt[i];
        if (vnew2 <= 0.0) {
            excess_c[i] = 0.5 * (sqr(vr) + sqr(vt) - vnew2) * m;
            event = true;
        } else {
            excess_c[i] = -1.0;
            double alpha = sqrt(vnew2 / (sqr(vr) + sqr(vt)));
            vr *= alpha;
            vt *= alpha;
            f.vr[i] = vr; f.vt[i] = vt;
            f.vrnew[i] = vr; f.vtnew[i] = vt;      // post-scaling values, read by the chain
        }
    }
    const uint64_t bal = __ballot(event);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) wcnt[w] = (int)__popcll(bal);
    __syncthreads();
    int pos = 0, cnt = 0;
    for (int q = 0; q < GT / 64; q++) {
        if (q < w) pos += wcnt[q];
        cnt += wcnt[q];
    }
    if (threadIdx.x == 0) blk_cnt[kg_.bid] = cnt;
    if (blk_events && event)               // a block's events from its first star's place on
        blk_events[(int64_t)kg_.bid * GT + pos + __popcll(bal & ((1ull << lane) - 1ull))] = i;
}
};

// Exclusive scan of the per-block event counts, in place, and their total.  A wave takes a
// contiguous range in rows of 64, held in registers when there are at most SV3_ROWS (so the
// write-back waits on no load); the ranges' sums go through LDS.  (With a range per thread the
// loads and stores were 128 bytes apart: 18 us for 15625 counts, now 11.)
constexpr int SV3_ROWS = 16;
struct sv3_scan_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s, int64_t *__restrict__ blk_cnt, int64_t nb,
                                               int64_t *__restrict__ relink)
{
    __shared__ int wtot[16];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int64_t rows = ((nb + 15) / 16 + 63) / 64, b0 = w * rows * 64 + lane;
    const bool regs = rows <= SV3_ROWS;
    int v[SV3_ROWS];
    int sum = 0;
    if (regs) {
#pragma unroll
        for (int q = 0; q < SV3_ROWS; q++) {
            v[q] = q < rows && b0 + q * 64 < nb ? (int)blk_cnt[b0 + q * 64] : 0;
            sum += v[q];
        }
    } else {
        for (int64_t q = 0; q < rows; q++)
            if (b0 + q * 64 < nb) sum += (int)blk_cnt[b0 + q * 64];
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) sum += __shfl_xor(sum, d, 64);
    if (lane == 0) wtot[w] = sum;
    __syncthreads();
    int64_t run = 0, tot = 0;                  // before the row in hand; of all
    for (int q = 0; q < 16; q++) {
        if (q < w) run += wtot[q];
        tot += wtot[q];
    }
    if (t == 0) {
        s->n_excess = tot;
        *relink = INT64_MAX;                   // sv3_verify_kernel takes the minimum
    }
    auto row = [&](int64_t q, int c) {
        int inc = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(inc, d, 64);
            if (lane >= d) inc += o;
        }
        if (b0 + q * 64 < nb) blk_cnt[b0 + q * 64] = run + inc - c;
        run += __shfl(inc, 63, 64);
    };
    if (regs) {
#pragma unroll
        for (int q = 0; q < SV3_ROWS; q++)
            if (q < rows) row(q, v[q]);
    } else {
        for (int64_t q = 0; q < rows; q++) row(q, b0 + q * 64 < nb ? (int)blk_cnt[b0 + q * 64] : 0);
    }
}
};

// ordered list of the event stars
struct sv3_compact_kernel {
    static constexpr int LB = GT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s, const double *__restrict__ excess_c,
                                                         const int64_t *__restrict__ blk_off,
                                                         int64_t *__restrict__ events)
{
    __shared__ int wcnt[GT / 64];
    int64_t i = 1 + (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    bool ev = i <= s->n_max && excess_c[i] >= 0.0;
    uint64_t bal = __ballot(ev);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) wcnt[w] = __popcll(bal);
    __syncthreads();
    int64_t pos = blk_off[kg_.bid];
    for (int w2 = 0; w2 < w; w2++) pos += wcnt[w2];
    pos += __popcll(bal & ((1ull << lane) - 1ull));
    if (ev) events[pos] = i;
}
};

constexpr int64_t SPEC_WALK_MAX = 4096;

// One episode of the excess chain starting at event star `i` with no excess
// carried into it: event stars add their excess, the other stars absorb
// min(0.8 KE, excess) each (cmc_utils.c:268-310).  Returns the star at which the
// excess reaches 0, n + 1 when excess is left at the end (dropped at one rank,
// cmc_utils.c:313-353), or -1 after `max_steps` stars.
__device__ int64_t excess_walk(const DevFields &f, const double *__restrict__ excess_c, int64_t i, int64_t n,
                               bool write, int64_t max_steps)
{
    const double E_dump_factor = 0.8;
    double Eexcess = 0.0;
    for (int64_t steps = 0; i <= n; i++, steps++) {
        if (steps >= max_steps) return -1;
        double c = excess_c[i];
        if (c >= 0.0) {
            Eexcess += c;
        } else if (Eexcess > 0) {
            double m = f.m[i], vr = f.vrnew[i], vt = f.vtnew[i];
            double v2 = sqr(vr) + sqr(vt);
            double E_dump_capacity = E_dump_factor * 0.5 * m * v2;
            double E_dump = E_dump_capacity <= Eexcess ? E_dump_capacity : Eexcess;
            if (write) {
                double exc_ratio = sqrt((v2 - 2 * E_dump / m) / v2);
                f.vr[i] = vr * exc_ratio;
                f.vt[i] = vt * exc_ratio;
            }
            Eexcess -= E_dump;
        }
        if (!(Eexcess > 0)) return i;
    }
    return n + 1;
}

// The same by a whole wave, unbounded: 64 stars' values at a time in its lanes, so that the
// chain of additions waits on no memory.  Every lane returns the end.  (With the relinking of
// 64 heads at a time, set_velocities3 with 1% / 30% of events: 2.15 -> 1.05 / 55 -> 16 ms at
// N = 1e6, 0.31 -> 0.19 / 15 -> 4.6 at 3e5.)
__device__ __forceinline__ double wave_value(double x, int lane)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, lane), hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ int64_t wave_value(int64_t x, int lane)
{
    return __double_as_longlong(wave_value(__longlong_as_double(x), lane));
}
template <bool WRITE>
__device__ __forceinline__ int64_t excess_walk_wave(const DevFields &f, const double *__restrict__ excess_c, int64_t i, int64_t n)
{
    const double E_dump_factor = 0.8;
    const int lane = threadIdx.x & 63;
    double Eexcess = 0.0;
    for (; i <= n; i += 64) {
        const int cnt = n - i < 63 ? (int)(n - i) + 1 : 64;
        const int64_t k = i + (lane < cnt ? lane : cnt - 1);
        const double c = excess_c[k], m = f.m[k], vr = f.vrnew[k], vt = f.vtnew[k];
        const double v2 = sqr(vr) + sqr(vt);
        const double capacity = E_dump_factor * 0.5 * m * v2;
        double dumped = -1.0;                      // this lane's star: what it absorbs
        int q = 0;
        for (; q < cnt; q++) {
            const double cq = wave_value(c, q);
            if (cq >= 0.0) {
                Eexcess += cq;
            } else if (Eexcess > 0) {
                const double cap = wave_value(capacity, q), E_dump = cap <= Eexcess ? cap : Eexcess;
                if (lane == q) dumped = E_dump;
                Eexcess -= E_dump;
            }
            if (!(Eexcess > 0)) break;
        }
        if (WRITE && dumped >= 0.0) {
            const double exc_ratio = sqrt((v2 - 2 * dumped / m) / v2);
            f.vr[k] = vr * exc_ratio;
            f.vt[k] = vt * exc_ratio;
        }
        if (q < cnt) return i + q;
    }
    return n + 1;
}

// Fresh (no carried excess) bounded walk of every event.  joins[d] = 1 when that
// walk reaches event d + 1 or was cut off, so event d + 1 is presumed to lie inside
// the same episode.  An episode starting at a true head is exactly its fresh walk.
__device__ __forceinline__ void sv3_spec(const DevFields &f, const double *__restrict__ excess_c, const int64_t *events,
                                         int64_t *wend, int32_t *joins, int64_t n, int64_t ne, int64_t d0, int64_t stride,
                                         int64_t max_steps = SPEC_WALK_MAX)
{
    for (int64_t d = d0; d < ne; d += stride) {
        int64_t e = excess_walk(f, excess_c, events[d], n, false, max_steps);
        wend[d] = e;
        joins[d] = (e < 0) || (d + 1 < ne && e >= events[d + 1]);
    }
}
struct sv3_spec_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, const double *__restrict__ excess_c,
                                const int64_t *__restrict__ events, int64_t *__restrict__ wend,
                                int32_t *__restrict__ joins)
{
    sv3_spec(f, excess_c, events, wend, joins, s->n_max, s->n_excess, (int64_t)kg_.bid * blockDim.x + threadIdx.x,
             (int64_t)kg_.nb * blockDim.x);
}
};

// Presumed heads are d = 0 and every d with joins[d-1] = 0; the presumed group of
// head d runs to the first q >= d with joins[q] = 0.  If every presumed head's walk
// ends inside its group's span [events[q], events[q+1]), then by induction from
// event 0 (which starts with no carried excess) each presumed head is a true head
// and its walk is the true episode.  Otherwise the heads are relinked exactly.
__device__ __forceinline__ void sv3_verify(const int64_t *events, const int32_t *joins, const int64_t *wend, int64_t *relink,
                                           int64_t ne, int64_t d0, int64_t stride)
{
    for (int64_t d = d0; d < ne; d += stride) {
        if (d > 0 && joins[d - 1]) continue;
        int64_t q = d;
        while (q + 1 < ne && joins[q]) q++;
        int64_t e = wend[d];
        if (e < 0 || e < events[q] || (q + 1 < ne && e >= events[q + 1]))
            atomicMin((unsigned long long *)relink, (unsigned long long)d);
    }
}
struct sv3_verify_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s, const int64_t *__restrict__ events,
                                  const int32_t *__restrict__ joins, const int64_t *__restrict__ wend,
                                  int64_t *__restrict__ relink)
{
    sv3_verify(events, joins, wend, relink, s->n_excess, (int64_t)kg_.bid * blockDim.x + threadIdx.x,
               (int64_t)kg_.nb * blockDim.x);
}
};

// Exact head chain in event order: the next head is the first event after the end
// of the current episode.  Runs only when a presumed head failed the check, and
// starts at the first one that did: every presumed head before it passed, so by
// induction it is a true head and the groups before it are exact.  One whole wave: 64 events
// and the ends of their own walks in its lanes.
__device__ __forceinline__ void sv3_relink(const DevFields &f, const double *__restrict__ excess_c, const int64_t *events,
                                           int64_t *wend, int32_t *joins, int64_t first, int64_t n, int64_t ne)
{
    const int lane = threadIdx.x & 63;
    int64_t end = -1;                              // of the episode in hand
    for (int64_t base = first; base < ne; base += 64) {
        const bool live = base + lane < ne;
        const int64_t ev = live ? events[base + lane] : INT64_MAX, we = live ? wend[base + lane] : 0;
        const int cnt = ne - base < 64 ? (int)(ne - base) : 64;
        uint64_t heads = 0;
        for (int l = 0;; l++) {
            l += (int)__popcll(__ballot(lane >= l && ev <= end));      // the next events up to its end
            if (l >= cnt) break;
            heads |= 1ull << l;
            end = wave_value(we, l);
            if (end < 0) {
                end = excess_walk_wave<false>(f, excess_c, wave_value(ev, l), n);
                if (lane == l) wend[base + l] = end;
            }
        }
        if (live && base + lane > first) joins[base + lane - 1] = (heads >> lane) & 1 ? 0 : 1;
    }
}
struct sv3_relink_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, const double *__restrict__ excess_c,
                                  const int64_t *__restrict__ events, int64_t *__restrict__ wend,
                                  int32_t *__restrict__ joins, const int64_t *__restrict__ relink)
{
    sv3_relink(f, excess_c, events, wend, joins, *relink, s->n_max, s->n_excess);
}
};

// Every head walks its episode and writes the dumped velocities: short episodes a thread
// each, the long ones a wave (every wave of the block calls; d0: the thread's first event).
constexpr int64_t LONG_EPISODE = 256;
__device__ __forceinline__ void sv3_heads(const DevFields &f, const double *__restrict__ excess_c, const int64_t *events,
                                          const int32_t *joins, const int64_t *wend, int64_t n, int64_t ne, int64_t d0,
                                          int64_t stride)
{
    const int lane = threadIdx.x & 63;
    for (int64_t d = d0; d - lane < ne; d += stride) {     // wave-uniform
        const bool head = d < ne && (d == 0 || !joins[d - 1]);
        const int64_t i = head ? events[d] : 0;
        const bool lng = head && (wend[d] < 0 || wend[d] - i >= LONG_EPISODE);
        if (head && !lng) excess_walk(f, excess_c, i, n, true, INT64_MAX);
        for (uint64_t todo = __ballot(lng); todo; todo &= todo - 1) {
            const int src = __ffsll((unsigned long long)todo) - 1;
            excess_walk_wave<true>(f, excess_c, wave_value(i, src), n);
        }
    }
}
struct sv3_heads_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, const double *__restrict__ excess_c,
                                 const int64_t *__restrict__ events, const int32_t *__restrict__ joins,
                                 const int64_t *__restrict__ wend)
{
    sv3_heads(f, excess_c, events, joins, wend, s->n_max, s->n_excess, (int64_t)kg_.bid * blockDim.x + threadIdx.x,
              (int64_t)kg_.nb * blockDim.x);
}
};

// The excess chain after sv3_kernel (the count of events, their ordered list, and the four
// kernels on it above) in one block for a cluster of at most SV3_ONE stars: six launches of
// 1 to 4 us with gaps as long.  The list comes from those of sv3_kernel's blocks.  (Without
// events set_velocities3 takes 47 us at N = 6e4, 75 by the launches; with 1% of them 70 / 75,
// with 30% 7.1 / 7.4 ms.)
constexpr int64_t SV3_ONE = 65536;
struct sv3_one_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, const double *__restrict__ excess_c,
                                               const int64_t *__restrict__ blk_cnt, int nb, int64_t *events, int64_t *wend,
                                               int32_t *joins, const int64_t *__restrict__ blk_events)
{
    constexpr int NB = SV3_ONE / GT, NW = NB / 64;     // as many waves scan the counts
    __shared__ int off[NB + 1], wtot[NW];
    __shared__ int64_t relink;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int64_t n = s->n_max;
    if (t < NB) {
        const int c = t < nb ? (int)blk_cnt[t] : 0;
        int inc = c;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(inc, d, 64);
            if (lane >= d) inc += o;
        }
        off[t] = inc - c;
        if (lane == 63) wtot[w] = inc;
    }
    __syncthreads();
    int ne = 0;
    for (int q = 0; q < NW; q++) {
        if (q == w && t < NB) off[t] += ne;
        ne += wtot[q];
    }
    ne = __builtin_amdgcn_readfirstlane(ne);       // scalars: the walks' branches depend on them
    if (t == 0) {
        off[NB] = ne;
        s->n_excess = ne;
        relink = INT64_MAX;
    }
    if (ne == 0) return;
    __syncthreads();
    for (int e = t; e < ne; e += 1024) {           // event e is number e - off[b] of its block b
        int b = 0, hi = nb - 1;
        while (b < hi) {
            const int m = (b + hi + 1) >> 1;
            if (off[m] <= e) b = m;
            else hi = m - 1;
        }
        events[e] = blk_events[(int64_t)b * GT + (e - off[b])];
    }
    __threadfence_block();
    __syncthreads();
    // one compute unit's walks share its loads: with more events than threads they are cut off
    // sooner, and the exact chain goes on from there
    const int per = (ne + 1023) / 1024;
    sv3_spec(f, excess_c, events, wend, joins, n, ne, t, 1024, per > 1 ? SPEC_WALK_MAX / 8 / per : SPEC_WALK_MAX);
    __threadfence_block();
    __syncthreads();
    sv3_verify(events, joins, wend, &relink, ne, t, 1024);
    __syncthreads();
    if (t < 64) sv3_relink(f, excess_c, events, wend, joins, wave_value(relink, 0), n, ne);
    __threadfence_block();
    __syncthreads();
    sv3_heads(f, excess_c, events, joins, wend, n, ne, t, 1024);
}
};

struct energy_kernel {
    static constexpr int LB = GT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P,
                                                    double *__restrict__ partials)
{
    int64_t i = 1 + (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    double v[2] = {0.0, 0.0};
    int64_t n = s->n_max;
    if (i <= n) {
        double vr = f.vr[i], vt = f.vt[i], ph = f.phi[i], m = f.m[i];
        f.E[i] = ph + 0.5 * (sqr(vr) + sqr(vt));
        f.J[i] = f.r[i] * vt;
        v[0] = 0.5 * (sqr(vr) + sqr(vt)) * m * P.madhoc;
        v[1] = ph * m * P.madhoc + f.phi[0] * P.cenma_m * P.madhoc / n;
    }
    block_sum_store<2>(v, partials + 8 * kg_.bid);
}
};

// compute_energy_new (cmc_utils.c:2017-2028) + the totals of ComputeEnergy (and the step's end)
struct energy_end_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s, const double *__restrict__ partials, int64_t nblocks,
                                               bool end_step)
{
    double res[2];
    final_sum<2>(partials, nblocks, res);
    if (threadIdx.x == 0) {
        s->Eescaped += s->Eescaped_old;
        s->Jescaped += s->Jescaped_old;
        s->Etidal += s->Etidal_old;
        double K = res[0], Pt = res[1] * 0.5;
        s->Ekin = K;
        s->Epot = Pt;
        s->Etot = K + Pt + 0.0 + 0.0;
        s->Etot += 0.0 + s->Eescaped + 0.0 + 0.0;
        if (end_step) s->step += 1;
    }
}
};

unsigned grid_for(int64_t n) { return (unsigned)((n + GT - 1) / GT > 0 ? (n + GT - 1) / GT : 1); }
} // namespace

hipError_t launch_energy_conservation1(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub,
                                       hipStream_t st)
{
    kl<ec1_kernel>(dim3(grid_for(n_ub)), dim3(GT), 0, st, f, s, P);
    return hipGetLastError();
}
hipError_t launch_energy_conservation2(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub,
                                       hipStream_t st, bool with_ie, double *dpre, int32_t *strip_done, double *apo_max)
{
    if (with_ie && !dpre) return hipErrorInvalidValue;
    if (with_ie) kl<ec2_ie_kernel>(dim3(grid_for(n_ub)), dim3(GT), 0, st, f, s, P, dpre, strip_done, apo_max);
    else kl<ec2_kernel>(dim3(grid_for(n_ub)), dim3(GT), 0, st, f, s, P);
    return hipGetLastError();
}
hipError_t launch_strip(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc, int32_t *done,
                        int64_t n_ub, int passes, bool begin, hipStream_t st, const double *apo_max)
{
    (void)n_ub;
    // a fixed grid (grid-stride over the stars) that the per-block partials hold
    const unsigned nb = STRIP_BLOCKS;              // the scratch holds at least STRIP_BLOCKS partials
    if (sc.max_blocks < STRIP_BLOCKS) return hipErrorInvalidValue;
    if (begin) kl<strip_begin_kernel>(dim3(1), dim3(1), 0, st, s, done);
    for (int it = 0; it < passes; it++) {
        kl<strip_pass_kernel>(dim3(nb), dim3(GT), 0, st, f, s, P, (const int32_t *)done, sc.partials, apo_max);
        kl<strip_end_kernel>(dim3(1), dim3(GT), 0, st, s, P, done, (const double *)sc.partials, nb);
    }
    return hipGetLastError();
}

bool strip_one_block(int64_t n_ub) { return n_ub <= STRIP_ONE; }

// The loop whose begin energy_conservation2 has done, in one block: as many passes as the grid
// passes and the tail of a captured step have, or the eager loop.
hipError_t launch_strip_loop(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc, bool graph, hipStream_t st,
                             const double *apo_max)
{
    kl<strip_one_kernel>(dim3(1), dim3(STRIP_ONE_T), 0, st, f, s, P, sc.strip_done,
                         graph ? STRIP_GRAPH_PASSES + STRIP_TAIL_PASSES : 100002, graph, apo_max);
    return hipGetLastError();
}

hipError_t launch_strip_tail(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc, hipStream_t st,
                             const double *apo_max)
{
    if (sc.max_blocks < STRIP_BLOCKS) return hipErrorInvalidValue;
    kl<strip_tail_kernel>(dim3(1), dim3(GT), 0, st, f, s, P, sc.strip_done, sc.partials,
                       (unsigned)STRIP_BLOCKS, apo_max);
    return hipGetLastError();
}
hipError_t launch_intermediate_energy(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub,
                                      hipStream_t st)
{
    (void)P;
    kl<ie_kernel>(dim3(grid_for(n_ub)), dim3(GT), 0, st, f, s);
    return hipGetLastError();
}
hipError_t launch_ie_transfer(const DevFields &f, DevScalars *s, int64_t n_ub, hipStream_t st)
{
    kl<ie_transfer_kernel>(dim3(grid_for(n_ub)), dim3(GT), 0, st, f, s);
    return hipGetLastError();
}
hipError_t launch_set_velocities3(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc,
                                  int64_t n_ub, hipStream_t st, const double *r_old_sorted, const double *dpre)
{
    if ((r_old_sorted != nullptr) != (dpre != nullptr)) return hipErrorInvalidValue;
    int64_t nb = grid_for(n_ub);
    if (nb > sc.max_blocks) return hipErrorInvalidValue;
    unsigned ge = grid_for(n_ub);
    if (ge > 256) ge = 256;            // the excess-list kernels stride over the list
    // the step calls this right after the potential, which left the node table current
    if (!dpre)
        if (hipError_t e = launch_mid_build(f, s, sc, n_ub, st)) return e;
    if (r_old_sorted) {
        const int64_t mb = (n_ub + MERGE_BLK - 1) / MERGE_BLK;
        kl<old_node_potential_kernel>(dim3((unsigned)mb), dim3(MERGE_T), 0, st, r_old_sorted,
                                      (const double2 *)sc.nodes, s, sc.u_old, dpre);
    }
    // (the sort's records are free here)
    int64_t *blk_events = reinterpret_cast<int64_t *>(sc.sort_aos);
    kl<sv3_kernel>(dim3((unsigned)nb), dim3(GT), 0, st, f, s, P, sc.excess_c, sc.sv3_blk,
                       (const double2 *)sc.mid, (const double2 *)sc.nodes,
                       r_old_sorted ? (const double2 *)sc.u_old : nullptr, (const uint32_t *)sc.vals_a,
                       n_ub <= SV3_ONE ? blk_events : (int64_t *)nullptr);
    if (n_ub <= SV3_ONE) {
        kl<sv3_one_kernel>(dim3(1), dim3(1024), 0, st, f, s, (const double *)sc.excess_c, (const int64_t *)sc.sv3_blk, (int)nb,
                           sc.excess_list, sc.sv3_wend, sc.sv3_merged, (const int64_t *)blk_events);
        return hipGetLastError();
    }
    kl<sv3_scan_kernel>(dim3(1), dim3(1024), 0, st, s, sc.sv3_blk, nb, sc.sv3_fallback);
    kl<sv3_compact_kernel>(dim3((unsigned)nb), dim3(GT), 0, st, s, (const double *)sc.excess_c,
                       (const int64_t *)sc.sv3_blk, sc.excess_list);
    kl<sv3_spec_kernel>(dim3(ge), dim3(GT), 0, st, f, s, (const double *)sc.excess_c,
                       (const int64_t *)sc.excess_list, sc.sv3_wend, sc.sv3_merged);
    kl<sv3_verify_kernel>(dim3(ge), dim3(GT), 0, st, s, (const int64_t *)sc.excess_list,
                       (const int32_t *)sc.sv3_merged, (const int64_t *)sc.sv3_wend, sc.sv3_fallback);
    kl<sv3_relink_kernel>(dim3(1), dim3(64), 0, st, f, s, (const double *)sc.excess_c,
                       (const int64_t *)sc.excess_list, sc.sv3_wend, sc.sv3_merged, (const int64_t *)sc.sv3_fallback);
    kl<sv3_heads_kernel>(dim3(ge), dim3(GT), 0, st, f, s, (const double *)sc.excess_c,
                       (const int64_t *)sc.excess_list, (const int32_t *)sc.sv3_merged, (const int64_t *)sc.sv3_wend);
    return hipGetLastError();
}
hipError_t launch_compute_energy(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc,
                                 int64_t n_ub, hipStream_t st, bool end_step)
{
    int64_t nb = grid_for(n_ub);
    if (nb > sc.max_blocks) return hipErrorInvalidValue;
    kl<energy_kernel>(dim3((unsigned)nb), dim3(GT), 0, st, f, s, P, sc.partials);
    kl<energy_end_kernel>(dim3(1), dim3(GT), 0, st, s, (const double *)sc.partials, nb, end_step);
    return hipGetLastError();
}
