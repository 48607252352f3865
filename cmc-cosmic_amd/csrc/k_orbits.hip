// a5-a8: get_positions_loop (src/cmc/cmc_evolution_thr.c:784-937) with
// calc_orbit_new (src/cmc/cmc_orbit.c:413-540), find_zero_Q (src/cmc/cmc_nr.c:316-383),
// find_root_vr (:500-603) and potential(r) (src/cmc/cmc_utils.c:112-165).
//
// One thread per star.  The rejection loop's potential(r) bisection is narrowed to
// [kmin, kmax+1] (the bracket the apsides already bound; the result index is the
// same as the reference's full-range FindZero_r, see potential_at).  Each star draws
// from its own taus113 substream (offset step*2^72 + 2^70 + slot*2^20).
//
// get_positive_Q_index (cmc_orbit.c:30-59) scans linearly from the centre when Q at
// the star's own index is not positive (v_r rounded to ~0).  That O(N) walk by one
// thread would stall the whole phase, so such stars are deferred: a grid-wide
// search finds the same first positive index, and a tail kernel finishes them.
//
// The phase is bound about equally by vector instructions (4000 a wave, 56% of the sampler's
// time at N = 4e6), by the rate of gathers into the sorted (r, phi) table (16 B a node, a line
// each: about 5 a search and 4 a try), which at N = 4e6 is 64 MB and lives in L2/MALL, and by
// the gathers' latency; the compulsory HBM traffic is 96 B/star.  Sampler at N = 4e6: 1071 us
// with about 12 gathers a search and 6 a try, 873 with these, 787 with division-free signs,
// two-digit jumps and the tries' results through LDS instead of 5700 instructions a wave.
#include "kernels.hpp"

namespace {
constexpr int ORB_THREADS = 256;
constexpr int ORB_COARSE = 1024;     // LDS samples of the (r, phi) table per block

// Per-block partials of the orbit phase (fixed-order wave-shuffle tree, then the
// four waves in order): [0] max_r (max), [1] Eescaped, [2] Jescaped,
// [3] TidalMassLoss, [4] Etidal, [5..10] star counts by outcome (circular,
// removed E >= 0, removed r_apo >= Rtidal, destroyed, Brent, linear scan),
// [11] tries, [12] max tries (max), [13] learned brackets used, [14] learned
// brackets rejected.
constexpr int NRED = 15, RED_STRIDE = 16;
__device__ __forceinline__ bool red_is_max(int i) { return i == 0 || i == 12; }

// The counts come from ballots and the removed stars' sums are formed only in waves that
// have some (zeros add nothing), so a wave shuffles one value, not fifteen.
template <int THREADS>
__device__ void block_reduce_store(double max_r, double Em, double Jm, double mm, int flags, int ntry, int hits, int misses,
                                   double *__restrict__ out)
{
    __shared__ double wsum[THREADS / 64][NRED];
    const int w = threadIdx.x >> 6;
    const bool first = (threadIdx.x & 63) == 0;
    auto count = [](bool b) { return (int)__popcll(__ballot(b)); };
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(max_r, off);
        max_r = max_r >= o ? max_r : o;
    }
    if (__ballot(flags & (CMCG_SF_REMOVED_E | CMCG_SF_REMOVED_RT)))
        for (int off = 32; off > 0; off >>= 1) {
            Em += __shfl_xor(Em, off);
            Jm += __shfl_xor(Jm, off);
            mm += __shfl_xor(mm, off);
        }
    int sum = 0, top = 0, bits = 0;            // tries: sum and maximum over the wave, bit by bit
    for (; __ballot((ntry >> bits) != 0); bits++) sum += count((ntry >> bits) & 1) << bits;
    uint64_t at_top = ~0ull;
    while (bits-- > 0) {
        const uint64_t m = at_top & __ballot((ntry >> bits) & 1);
        if (m) { at_top = m; top |= 1 << bits; }
    }
    const int c[NRED - 5] = {count(flags & CMCG_SF_CIRCULAR),   count(flags & CMCG_SF_REMOVED_E),
                             count(flags & CMCG_SF_REMOVED_RT), count(flags & CMCG_SF_DESTROYED),
                             count(flags & CMCG_SF_BRENT),      count(flags & CMCG_SF_LINSCAN),
                             sum, top, count(hits & 1) + 2 * count(hits & 2), count(misses & 1) + 2 * count(misses & 2)};
    if (first) {
        wsum[w][0] = max_r;
        wsum[w][1] = Em; wsum[w][2] = Jm; wsum[w][3] = mm; wsum[w][4] = Em;
        for (int i = 5; i < NRED; i++) wsum[w][i] = (double)c[i - 5];
    }
    __syncthreads();
    if (threadIdx.x < NRED) {
        const int i = threadIdx.x;
        double a = wsum[0][i];
        for (int k = 1; k < THREADS / 64; k++) a = red_is_max(i) ? (a >= wsum[k][i] ? a : wsum[k][i]) : a + wsum[k][i];
        out[i] = a;
    }
}

// outcome counters of one deferred star into its record (its scan is counted where it was deferred)
__device__ __forceinline__ void count_star(double (&red)[NRED], int flags, int ntry, int hits, int misses)
{
    red[5] += (flags & CMCG_SF_CIRCULAR) ? 1.0 : 0.0;
    red[6] += (flags & CMCG_SF_REMOVED_E) ? 1.0 : 0.0;
    red[7] += (flags & CMCG_SF_REMOVED_RT) ? 1.0 : 0.0;
    red[8] += (flags & CMCG_SF_DESTROYED) ? 1.0 : 0.0;
    red[9] += (flags & CMCG_SF_BRENT) ? 1.0 : 0.0;
    red[11] += (double)ntry;
    red[12] = red[12] >= (double)ntry ? red[12] : (double)ntry;
    red[13] += (double)hits;
    red[14] += (double)misses;
}

// remove_star (cmc_evolution_thr.c:655-716) contributions: Eescaped, Jescaped,
// TidalMassLoss, Etidal
__device__ __forceinline__ void removed(double (&red)[NRED], double Ej, double J, double mj, const KParams &P)
{
    red[1] = Ej * mj / (double)P.n_star;
    red[2] = J * mj / (double)P.n_star;
    red[3] = mj / (double)P.n_star;
    red[4] = Ej * mj / (double)P.n_star;
}

// DevFields::knew of a star that stays at r_j (a circular orbit): the nodes below it
template <class N>
__device__ __forceinline__ int32_t nodes_below(const N &nd, int64_t j, double rj)
{
    int64_t k = j - 1;
    while (k > 0 && !(nd.R(k) < rj)) k--;
    return (int32_t)k;
}
// ... and of one sampled at x between nodes k and k + 1 (the sort drops radii at or beyond SF_INFINITY)
__device__ __forceinline__ int32_t knew_of(int32_t k, double x) { return x < CMCG_SF_INFINITY ? k : -1; }

// The part of get_positions_loop after the positive-Q index is known
// (cmc_evolution_thr.c:832-934).
template <class N>
__device__ void sample_star(const N &nd, const DevFields &f, DevScalars *s, const KParams &P, Rng rng,
                            int64_t n, int64_t j, double rj, double mj, double E,
                            double Ej, double J, int64_t ktemp, int &flags, int &ntry, int &hits, int &misses,
                            double (&red)[NRED])
{
    const double *__restrict__ r = f.r;
    const double *__restrict__ phi = f.phi;
    OrbitRS o = calc_orbit_from_n(nd, r, phi, n, j, rj, mj, P, E, J, ktemp);
    if (o.err) dev_set_error(s, o.err, j);
    hits = o.hint_hits;
    misses = o.hint_misses;
    if (o.brent) flags |= CMCG_SF_BRENT;
    if (o.circular) {
        f.rnew[j] = rj; f.vrnew[j] = f.vr[j]; f.vtnew[j] = f.vt[j];
        f.knew[j] = nodes_below(nd, j, rj);
        flags |= CMCG_SF_CIRCULAR;
        return;
    }
    if (o.ra >= s->Rtidal) {
        f.r_apo[j] = o.ra; f.r_peri[j] = o.rp;
        f.rnew[j] = CMCG_SF_INFINITY; f.vrnew[j] = 0.0; f.vtnew[j] = 0.0;
        f.knew[j] = -1;
        removed(red, Ej, J, mj, P);
        flags |= CMCG_SF_REMOVED_RT;
        return;
    }
    const double rmin = o.rp, rmax = o.ra;
    double g1 = sqrt(3.0 * (rmax - rmin) / o.dQdrp);
    double g2 = sqrt(-3.0 * (rmax - rmin) / o.dQdra);
    double F = 1.2 * (g1 >= g2 ? g1 : g2);
    // narrowed bracket for potential(r): r in [rmin, rmax] within [r_kmin, r_kmax+1]
    int64_t lo0 = o.kmin < 1 ? 1 : o.kmin;
    int64_t hi0 = o.kmax + 1 > n + 1 ? n + 1 : o.kmax + 1;
    const double r_lo0 = nd.R(lo0), r_hi0 = nd.R(hi0);
    double X = 0.0, rr = 0.0, vr = 0.0, potr = 0.0;
    int k;
    int32_t kn = 0;
    bool bad = false;
    for (k = 1; k <= CMCG_N_TRY; k++) {
        X = rng_dbl(rng);
        double s0 = 2.0 * X - 1.0;
        double g0 = F * rng_dbl(rng);
        rr = 0.5 * (rmin + rmax) + 0.25 * (rmax - rmin) * (3.0 * s0 - s0 * s0 * s0);
        int64_t lo = lo0, hi = hi0;
        if (!(r_lo0 < rr)) lo = 1;
        if (!(rr <= r_hi0)) hi = n + 1;
        potr = potential_at_n(nd, n, rr, lo, hi, &bad, &kn);
        double pot = potr + phi_s_own(rj, mj, P.inv_nstar, rr);
        double drds = 0.25 * (rmax - rmin) * (3.0 - 3.0 * s0 * s0);
        double Q = 2.0 * E - 2.0 * pot - J * J / rr / rr;
        if (Q >= 0.0) {
            vr = sqrt(Q);
        } else {
            if (isnan(Q)) { dev_set_error(s, CMCG_E_NAN, j); break; }
            vr = 0;
        }
        if (g0 < 1.0 / vr * drds) break;
    }
    if (bad) dev_set_error(s, CMCG_E_BRACKET, j);
    if (k == CMCG_N_TRY + 1) dev_set_error(s, CMCG_E_NTRY, j);
    ntry = k;
    f.X[j] = X;
    f.r_peri[j] = rmin;
    f.r_apo[j] = rmax;
    if (rng_dbl(rng) < 0.5) vr = -vr;
    f.rnew[j] = rr;
    f.knew[j] = knew_of(kn, rr);
    f.vrnew[j] = vr;
    f.vtnew[j] = J / rr;
    f.pot_rnew[j] = potr;
    flags |= 256;      // sampled: pot_rnew holds potential(rnew)
    red[0] = rr;
}

// ------------------------------------------------------------------ wave-parallel tries
// The rejection loop of get_positions_loop (cmc_evolution_thr.c:858-906) takes a
// geometric number of tries (mean ~2), so a wave that ran one star per lane would
// idle most lanes while its slowest star (~8 tries) finishes.  Instead the wave
// evaluates tries in rounds: the stars still trying share the 64 lanes, each lane
// taking the next untried try number of one star, stepped to that try's draws in the
// star's own substream (try t uses draws 2t-2 and 2t-1, the sign draw follows the
// accepted try).  A star's result is its lowest-numbered terminating try, exactly as
// the sequential loop, so outputs do not depend on the grouping.

// What a star's tries need (set by prepare_star), and in its place their result, written by
// the lane that ran the last one.
struct TryCtx {
    double rmin, rmax, F, E, rj, mj, J;
};
struct TryOut {
    double X, rr, vr, potr;
    int32_t kn;        // index of rr among the nodes
    int32_t k;         // tries taken; CMCG_N_TRY + 1 when none was accepted
    int32_t nan, pad;
    double J;          // TryCtx::J
};
union TrySlot {
    Rng rng;           // while the star's apsides are sought: its substream state, out of the registers
    TryCtx in;
    TryOut out;
};
static_assert(sizeof(TryCtx) == sizeof(TryOut) && offsetof(TryCtx, J) == offsetof(TryOut, J), "J is common to both");

// The part of get_positions_loop between the positive-Q index and the rejection loop
// (cmc_evolution_thr.c:832-857): apsides, removal at r_apo >= Rtidal, circular
// orbits, and the loop's constants.  Returns true if the star samples a new radius.
template <class N>
__device__ __forceinline__ bool prepare_star(const N &nd, const DevFields &f, DevScalars *s, const KParams &P,
                                             const Coarse &C, int64_t n, int64_t j, const QStar &q, double pj, int &flags, int &hits, int &misses,
                                             TrySlot &slot, Rng &rng)
{
    const double rj = q.rj;
    OrbitRS o = calc_orbit_core<N, true>(nd, f.r, f.phi, n, j, rj, q.mj, P, q.E, q.J, j, C, q, pj);
    if (o.err) dev_set_error(s, o.err, j);
    hits = o.hint_hits;
    misses = o.hint_misses;
    if (o.brent) flags |= CMCG_SF_BRENT;
    if (o.circular) {
        f.rnew[j] = rj; f.vrnew[j] = f.vr[j]; f.vtnew[j] = f.vt[j];
        f.knew[j] = nodes_below(nd, j, rj);
        flags |= CMCG_SF_CIRCULAR;
        return false;
    }
    if (o.ra >= s->Rtidal) {
        f.r_apo[j] = o.ra; f.r_peri[j] = o.rp;
        f.rnew[j] = CMCG_SF_INFINITY; f.vrnew[j] = 0.0; f.vtnew[j] = 0.0;
        f.knew[j] = -1;
        flags |= CMCG_SF_REMOVED_RT;      // its removal sums are added by the caller
        return false;
    }
    f.r_peri[j] = o.rp;
    f.r_apo[j] = o.ra;
    const double g1 = sqrt(3.0 * (o.ra - o.rp) / o.dQdrp);
    const double g2 = sqrt(-3.0 * (o.ra - o.rp) / o.dQdra);
    rng = slot.rng;
    TryCtx &tc = slot.in;
    tc.rmin = o.rp; tc.rmax = o.ra;
    tc.F = 1.2 * (g1 >= g2 ? g1 : g2);
    tc.E = q.E; tc.J = q.J; tc.rj = rj; tc.mj = q.mj;
    return true;
}

// One try (cmc_evolution_thr.c:862-886) from the state at its first draw; on return
// st is the state after the try's two draws.
__device__ __forceinline__ bool one_try(const double2 *__restrict__ nodes, const RIdx &ri, double r1, const KParams &P,
                                        int64_t n, const TryCtx &tc,
                                        Rng &st, double &X, double &rr, double &vr, double &potr, int32_t &kn,
                                        bool &bad, bool &nan)
{
    X = rng_dbl(st);
    const double s0 = 2.0 * X - 1.0;
    const double g0 = tc.F * rng_dbl(st);
    rr = 0.5 * (tc.rmin + tc.rmax) + 0.25 * (tc.rmax - tc.rmin) * (3.0 * s0 - s0 * s0 * s0);
    potr = potential_at_ridx(nodes, n, r1, rr, ri, &bad, &kn);
    const double pot = potr + phi_s_own(tc.rj, tc.mj, P.inv_nstar, rr);
    const double drds = 0.25 * (tc.rmax - tc.rmin) * (3.0 - 3.0 * s0 * s0);
    const double Q = 2.0 * tc.E - 2.0 * pot - tc.J * tc.J / rr / rr;
    if (Q >= 0.0) {
        vr = sqrt(Q);
    } else {
        if (isnan(Q)) { nan = true; vr = 0.0; return true; }
        vr = 0;
    }
    return g0 < 1.0 / vr * drds;
}

__device__ __forceinline__ uint32_t from_lane(uint32_t x, int lane4)
{
    return (uint32_t)__builtin_amdgcn_ds_bpermute(lane4, (int)x);
}

// All lanes of the wave call this together (convergent).  need: this lane's star
// samples; slots: the wave's 64 try constants in LDS (slot = lane, written before a
// block barrier), which hold the results on return; rng: this lane's substream state before
// its star's first try.  Returns whether a try up to the star's last found no interval.
// A round has R stars: c = 64 / R lanes each, one more for the first 64 - c R of them, but at
// most CAP (then the rest idle): fewer wasted tries.  About 3.4 rounds a wave at CAP = 4.
template <int CAP>
__device__ bool wave_tries(const double2 *__restrict__ nodes, const RIdx &ri, const KParams &P, int64_t n, bool need,
                           TrySlot *__restrict__ slots, Rng rng)
{
    const int lane = threadIdx.x & 63;
    int next = 1;                         // owner: first try not yet evaluated
    bool bad_acc = false;
    const double r1 = nodes[1].x;
    auto rank_in = [](uint64_t m) {       // set bits of m below the lane
        return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
    };
    // quotients of integers up to 64 by the reciprocal's estimate: a half keeps them off the integers
    auto over = [](float a, int b) { return (int)((a + 0.5f) * __builtin_amdgcn_rcpf((float)b)); };
    uint64_t pending = __ballot(need);
    while (pending) {
        const int R = (int)__popcll(pending), c64 = over(64.f, R);
        const int c = c64 >= CAP ? CAP : c64, rem = c64 >= CAP ? 0 : 64 - c64 * R;
        const bool owner = (pending >> lane) & 1ull;
        const int my_q = rank_in(pending);
        // lane q learns which lane owns the q-th star (the others fill the lanes after R)
        const int own = __builtin_amdgcn_ds_permute((owner ? my_q : R + lane - my_q) << 2, lane);
        const int big = (c + 1) * rem;
        const bool in_big = lane < big;
        const int cs = in_big ? c + 1 : c, l2 = in_big ? lane : lane - big;
        const int g = over((float)l2, cs), o = l2 - g * cs, q = in_big ? g : rem + g;
        const bool idle = q >= R;
        const int sl = (int)from_lane((uint32_t)own, idle ? 0 : q << 2), sl4 = sl << 2;   // owner of the star helped
        const TryCtx t = slots[sl].in;
        Rng st{from_lane(rng.z0, sl4), from_lane(rng.z1, sl4), from_lane(rng.z2, sl4), from_lane(rng.z3, sl4)};
        const int k = (int)from_lane((uint32_t)next, sl4) + o;
        const bool eval = !idle && k <= CMCG_N_TRY;
        if (!idle)
            for (int d = 0; d < 2 * o; d++) (void)rng_int(st);
        double X = 0.0, rr = 0.0, vr = 0.0, potr = 0.0;
        int32_t kn = 0;
        bool bad = false, nan = false, term = false;
        if (eval) {
            term = one_try(nodes, ri, r1, P, n, t, st, X, rr, vr, potr, kn, bad, nan);
            // the sign draw follows the accepted try, or the last one if the star runs out of them
            if ((term && !nan) || k == CMCG_N_TRY) {
                Rng sg = st;
                if (rng_dbl(sg) < 0.5) vr = -vr;
            }
        }
        // the star's lanes are [lane - o, lane - o + cs); its result is their first that ends
        const uint64_t tmask = __ballot(eval && term), bmask = __ballot(eval && bad);
        const uint64_t ones = cs >= 64 ? ~0ull : (1ull << cs) - 1ull;
        const uint64_t mine = (tmask >> (lane - o)) & ones;
        const bool win = eval && (term ? (mine & ((1ull << o) - 1ull)) == 0ull : (k == CMCG_N_TRY && mine == 0ull));
        if (win) {
            TryOut &r = slots[sl].out;
            r.X = X; r.rr = rr; r.vr = vr; r.potr = potr; r.kn = kn;
            r.k = term ? k : CMCG_N_TRY + 1;
            r.nan = nan;
        }
        const uint64_t wmask = __ballot(win);
        // owners: the star's lanes are [base, base + my_cs)
        const int my_cs = my_q < rem ? c + 1 : c;
        const int base = owner ? my_q * c + (my_q < rem ? my_q : rem) : 0;
        const uint64_t my_ones = my_cs >= 64 ? ~0ull : (1ull << my_cs) - 1ull;
        const uint64_t won = (wmask >> base) & my_ones;
        const bool done = owner && won != 0ull;
        if (bmask && owner) {              // up to the final try, or all of this round's
            const uint64_t upto = done ? ((won << 1) - 1ull) : my_ones;
            bad_acc |= ((bmask >> base) & my_ones & upto) != 0ull;
        }
        const int last4 = (base + my_cs - 1) << 2;
        const Rng ns{from_lane(st.z0, last4), from_lane(st.z1, last4), from_lane(st.z2, last4), from_lane(st.z3, last4)};
        if (owner && !done) {              // go on from the round's last try
            next += my_cs;
            rng = ns;
        }
        pending &= ~__ballot(done);
    }
    // the results come from other lanes of the wave
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    return bad_acc;
}

// Slot j draws from offset j 2^20 (base[2]: the state of slot 1): the wave jumps to its
// first slot, its lanes on through the LDS tables.  With learned brackets the network's
// prediction proposes both find_zero_Q brackets.
// MINB: blocks per CU the register allocation must allow (1: no constraint; 5 blocks of 256
// threads: five waves per SIMD, at most 102 registers)
template <int THREADS, int COARSE, int CAP, int MINB>
struct orbits_kernel {
    static constexpr int LB = THREADS, MB = MINB;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P,
                                                             const JumpTables *__restrict__ jump,
                                                             const Rng *__restrict__ base,
                                                             double *__restrict__ partials,
                                                             int64_t *__restrict__ defer_list,
                                                             int64_t *__restrict__ defer_kfirst,
                                                             const float2 *__restrict__ pred, float margin,
                                                             const double2 *__restrict__ nodes,
                                                             const double2 *__restrict__ coarse,
                                                             const uint32_t *__restrict__ ridx, int ridx_bits)
{
    // the jump table is needed only for the lanes' first states: the samples wait in
    // registers and take its place (31 KB in all: five blocks share a CU's 160 KB)
    __shared__ union alignas(16) Share {
        LaneDigit lt;
        struct { double cr[COARSE + 1], cphi[COARSE + 1]; } c;
    } sh;
    __shared__ TrySlot slot[THREADS];
    double *const cr = sh.c.cr, *const cphi = sh.c.cphi;
    const int64_t n = s->n_max;
    Coarse C;
    C.cr = cr; C.cphi = cphi; C.cs = COARSE; C.n1 = n + 1;
    C.stride = coarse_stride(n, COARSE);
    C.inv_stride = 0xffffffffu / (uint32_t)C.stride;
    C.hint = false; C.lrp = C.lra = 0.f; C.margin = margin;
    C.ri.t = nullptr;
    if (n >= 1) C.ri = ridx_of(ridx, nodes, n, ridx_bits);
    constexpr int NC = COARSE / THREADS;
    static_assert(COARSE % THREADS == 0, "the samples are dealt out evenly, and one more");
    double2 sample[NC];                        // built once per phase
#pragma unroll
    for (int u = 0; u < NC; u++) sample[u] = coarse[threadIdx.x + u * THREADS];
    {
        constexpr int NQ = (int)(sizeof(LaneDigit) / sizeof(uint4));
        const uint4 *src = reinterpret_cast<const uint4 *>(&jump->orbit.lo);
        uint4 *dst = reinterpret_cast<uint4 *>(&sh.lt);
        for (int q = threadIdx.x; q < NQ; q += THREADS) dst[q] = src[q];
    }
    const int64_t j = 1 + xcd_block(kg_) * blockDim.x + threadIdx.x;
    Rng rng = jump_uniform(jump->level + JL_SLOT + 1, JL_SLOT_N - 1, rng_uniform(base[2]),
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)((j - 1) >> 6)));
    __syncthreads();
    rng = jump_lane_digits(jump->orbit.hi, sh.lt, rng);
    slot[threadIdx.x].rng = rng;
    asm volatile("" ::: "memory");             // ... so that it is read again there
    __syncthreads();                           // the table is dead from here
#pragma unroll
    for (int u = 0; u < NC; u++) {
        cr[threadIdx.x + u * THREADS] = sample[u].x;
        cphi[threadIdx.x + u * THREADS] = sample[u].y;
    }
    if (threadIdx.x == 0) {
        const double2 last = coarse[COARSE];
        cr[COARSE] = last.x;
        cphi[COARSE] = last.y;
    }
    __syncthreads();
    bool need = false;
    int flags = 0, ntry = 0, hits = 0, misses = 0;
    if (j <= n) {
        const double rj = f.r[j], mj = f.m[j];
        const double Ej = f.E[j], J = f.J[j];
        const double E = Ej + phi_s_own(rj, mj, P.inv_nstar, rj);    // cmc_evolution_thr.c:806
        const QStar q = q_star(rj, mj, P.inv_nstar, E, J);
        if (mj < CMCG_ZERO) {
            // destroy_obj (cmc_dynamics_helper.c:131-153) + remove_star_center
            f.vr[j] = 0.0; f.vt[j] = 0.0; f.E[j] = 0.0; f.J[j] = 0.0; f.id[j] = 0;
            f.X[j] = 0.0; f.Y[j] = 0.0; f.r_peri[j] = 0.0; f.r_apo[j] = 0.0;
            f.rnew[j] = CMCG_SF_INFINITY; f.knew[j] = -1; f.m[j] = 2.2250738585072014e-308;
            f.vrnew[j] = 0.0; f.vtnew[j] = 0.0;
            flags = CMCG_SF_DESTROYED;
        } else if (E >= 0.0) {
            f.rnew[j] = CMCG_SF_INFINITY; f.vrnew[j] = 0.0; f.vtnew[j] = 0.0; f.knew[j] = -1;
            flags = CMCG_SF_REMOVED_E;
        } else {
            const double pj = f.phi[j];
            if (q_le0(q_sign(q, rj, pj))) {
                // linear-scan case: finished by the deferred path
                flags = CMCG_SF_LINSCAN;
                unsigned long long slot = atomicAdd((unsigned long long *)&s->n_defer, 1ull);
                if ((int64_t)slot < P.defer_cap) {
                    defer_list[slot] = j;
                    defer_kfirst[slot] = n + 2;          // the search takes the minimum
                } else {
                    dev_set_error(s, CMCG_E_STATE, j);
                }
            } else {
                if (pred) {
                    const float2 y = pred[j];
                    C.hint = true;
                    C.lrp = y.x;
                    C.lra = y.y;
                }
                need = prepare_star(PackedNodes{nodes}, f, s, P, C, n, j, q, pj, flags, hits, misses,
                                    slot[threadIdx.x], rng);
            }
        }
    }
    __syncthreads();                           // try constants visible to the wave
    // every lane of the wave takes part, stars or not
    const bool bad = wave_tries<CAP>(nodes, C.ri, P, n, need, slot + (threadIdx.x & ~63), rng);
    double max_r = 0.0, Em = 0.0, Jm = 0.0, mm = 0.0;
    if (j <= n) {
        if (need) {
            const TryOut to = slot[threadIdx.x].out;
            if (bad) dev_set_error(s, CMCG_E_BRACKET, j);
            if (to.nan) dev_set_error(s, CMCG_E_NAN, j);
            else if (to.k == CMCG_N_TRY + 1) dev_set_error(s, CMCG_E_NTRY, j);
            ntry = to.k;
            f.X[j] = to.X;
            f.rnew[j] = to.rr;
            f.knew[j] = knew_of(to.kn, to.rr);
            f.vrnew[j] = to.vr;
            f.vtnew[j] = to.J / to.rr;
            f.pot_rnew[j] = to.potr;
            flags |= 256;      // sampled: pot_rnew holds potential(rnew)
            max_r = to.rr;
        }
        if (flags & (CMCG_SF_REMOVED_E | CMCG_SF_REMOVED_RT)) {      // fields the removal left unchanged
            double red[NRED];
            removed(red, f.E[j], f.J[j], f.m[j], P);
            Em = red[1]; Jm = red[2]; mm = red[3];
        }
        f.flags[j] = flags;
        f.ntry[j] = ntry;
    }
    block_reduce_store<THREADS>(max_r, Em, Jm, mm, flags, ntry, hits, misses, partials + RED_STRIDE * xcd_block(kg_));
}
};

// The deferred stars in star order, so that the reduction of their sums does not depend on the
// order in which they were appended (one block): order[] is their stars and slots packed into
// one word, sorted.  A short list is sorted by one thread; a longer one by a bitonic sort over
// the next power of two (the list's capacity is one, above the number of stars), padded with
// INT64_MAX, in global memory.
constexpr int DEFER_T = 1024;
constexpr int DEFER_SLOT_BITS = 31;            // star and slot indices are below 2^31
__device__ __forceinline__ int64_t deferred(const DevScalars *s, const KParams &P)
{
    return s->n_defer < P.defer_cap ? s->n_defer : P.defer_cap;
}
__device__ void defer_sort(const int64_t *__restrict__ list, int64_t *__restrict__ order, int64_t nd)
{
    const int t = threadIdx.x;
    auto word = [&](int64_t d) { return (list[d] << DEFER_SLOT_BITS) | d; };
    if (nd <= 64) {
        if (t == 0)
            for (int64_t a = 0; a < nd; a++) {
                const int64_t v = word(a);
                int64_t b = a - 1;
                while (b >= 0 && order[b] > v) { order[b + 1] = order[b]; b--; }
                order[b + 1] = v;
            }
        return;
    }
    int64_t P = 1;
    while (P < nd) P <<= 1;
    for (int64_t i = t; i < P; i += DEFER_T) order[i] = i < nd ? word(i) : INT64_MAX;
    __syncthreads();
    for (int64_t k = 2; k <= P; k <<= 1)
        for (int64_t j = k >> 1; j > 0; j >>= 1) {
            for (int64_t i = t; i < P; i += DEFER_T) {
                const int64_t l = i ^ j;
                if (l > i) {
                    const int64_t a = order[i], b = order[l];
                    if ((a > b) == ((i & k) == 0)) { order[i] = b; order[l] = a; }
                }
            }
            __syncthreads();
        }
}

// Grid-wide equivalent of the linear scan: the first k in [0, N_MAX+1] with Q > 0 of every
// deferred star, four stars at a time, each by a quarter of the nb blocks.
__device__ void defer_search(const DevFields &f, const KParams &P, const int64_t *__restrict__ list,
                             int64_t *__restrict__ kfirst, int64_t nd, int64_t n, int b, int nb)
{
    const int64_t stride = (int64_t)(nb / 4) * DEFER_T;
    for (int64_t d = b & 3; d < nd; d += 4) {
        const int64_t j = list[d];
        const double rj = f.r[j], mj = f.m[j];
        const double E = f.E[j] + phi_s_own(rj, mj, P.inv_nstar, rj);
        const double J = f.J[j];
        for (int64_t k = (int64_t)(b >> 2) * DEFER_T + threadIdx.x; k <= n + 1; k += stride) {
            if (k > kfirst[d]) break;
            if (function_q(rj, mj, P.inv_nstar, f.r[k], f.phi[k], E, J) > 0.0)
                atomicMin((unsigned long long *)&kfirst[d], (unsigned long long)k);
        }
    }
}

// First level of the orbit phase's reduction: block B of RED2_BLOCKS sums the partial
// records of sampler blocks [B C, (B + 1) C), C = ceil(nblocks / RED2_BLOCKS); 16
// consecutive threads read one record (coalesced), its 64 groups take records
// g, g + 64, ... of the range, and the groups are combined in group order.
__device__ void orbits_part(const double *__restrict__ partials, int64_t nblocks, double *__restrict__ out, int B)
{
    __shared__ double gsum[64][RED_STRIDE];
    const int t = threadIdx.x, i = t & 15, g = t >> 4;
    const int64_t C = (nblocks + RED2_BLOCKS - 1) / RED2_BLOCKS;
    const int64_t b0 = (int64_t)B * C, b1 = b0 + C < nblocks ? b0 + C : nblocks;
    double acc = 0.0;
    if (i < NRED)
        for (int64_t b = b0 + g; b < b1; b += 64) {
            double p = partials[RED_STRIDE * b + i];
            acc = red_is_max(i) ? (acc >= p ? acc : p) : acc + p;
        }
    gsum[g][i] = acc;
    __syncthreads();
    if (t < NRED) {
        double a = gsum[0][t];
        for (int g2 = 1; g2 < 64; g2++) a = red_is_max(t) ? (a >= gsum[g2][t] ? a : gsum[g2][t]) : a + gsum[g2][t];
        out[RED_STRIDE * B + t] = a;
    }
}

// Whether the new radii's indices cut the stars into even buckets for the step's sort: up to
// BAL_MAX of them counted (one block).  A bucket is too long at twice its share and 10 more:
// what a sample can miss, 10 of 2048, costs its block less than 0.4 ms at N = 4e6.  (The
// deferred stars have the indices of their last orbits; counts decide only the speed.)
// Bound by one CU's misses, a line a sample: the kernel that holds this block takes 12.0 us at
// N = 4e6, as it does without the block; with 8192 samples and 40 more, 19.7.
constexpr int BAL_MAX = 2048;
__device__ void sort_balance(const int32_t *__restrict__ knew, int64_t n, int B, int32_t *uneven)
{
    __shared__ uint32_t hist[SB_MAX_BUCKETS];
    const int t = threadIdx.x, S = n < BAL_MAX ? (int)n : BAL_MAX;
    for (int b = t; b < B; b += DEFER_T) hist[b] = 0;
    const StepBucket bucket(n, B);
    const double stride = (double)n / (double)S;           // at least 1
    uint32_t k[BAL_MAX / DEFER_T];
#pragma unroll
    for (int u = 0; u < BAL_MAX / DEFER_T; u++) {
        const int q = u * DEFER_T + t;
        k[u] = q < S ? bucket(knew[1 + (int64_t)(q * stride)]) : (uint32_t)SB_TAIL;
    }
    __syncthreads();
    const uint32_t limit = 2 * (uint32_t)S / (uint32_t)B + 10;
    bool over = false;
#pragma unroll
    for (int u = 0; u < BAL_MAX / DEFER_T; u++)
        if (k[u] != SB_TAIL) over |= atomicAdd(&hist[k[u]], 1u) >= limit;
    if (over) *uneven = 2;
}
// Bucket boundaries from a sample of the new radii, for that case (one block).
__device__ void step_splits(const double *__restrict__ rnew, int64_t n, int B, uint64_t *__restrict__ split)
{
    __shared__ uint64_t key[SMP_MAX];
    const int t = threadIdx.x, S = n < SMP_MAX ? (int)n : SMP_MAX;
    for (int q = t; q < S; q += blockDim.x) {
        const double x = rnew[1 + (int64_t)q * n / S];
        key[q] = x < CMCG_SF_INFINITY ? sortable(x) : KEY_INF;
    }
    sample_sort(key, S);
    for (int b = t; b < B; b += blockDim.x) split[b] = b > 0 && S > 0 ? key[(int64_t)b * S / B] : 0ull;
}

// After the sampler, in one launch (three kernels of 4 to 12 us before): its reduction's first
// level, the order of the deferred stars, their linear scans, and the buckets' balance.
constexpr int DEFER_BLOCKS = 256;
struct after_orbits_kernel {
    static constexpr int LB = DEFER_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P,
                                                           const double *__restrict__ partials, int64_t nblocks,
                                                           double *__restrict__ red2, const int64_t *__restrict__ list,
                                                           int64_t *__restrict__ kfirst, int64_t *__restrict__ order,
                                                           int buckets, int32_t *uneven)
{
    const int b = (int)kg_.bid - RED2_BLOCKS - 1;
    if (b < -1) orbits_part(partials, nblocks, red2, (int)kg_.bid);
    else if (b == -1) defer_sort(list, order, deferred(s, P));
    else if (b == DEFER_BLOCKS) sort_balance(f.knew, s->n_max, buckets, uneven);
    else defer_search(f, P, list, kfirst, deferred(s, P), s->n_max, b, DEFER_BLOCKS);
}
};

// The deferred stars, ORB_THREADS at a time in list order, and the phase's sums: the
// sampler blocks' records (the first level's RED2_BLOCKS records, in block order), then
// each deferred star's in list (= star) order, as a single thread would add them; then
// the end of new_orbits_calculate.  Block 1: the step's bucket boundaries, where it needs them.
struct defer_tail_kernel {
    static constexpr int LB = ORB_THREADS, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P,
                                                                 const RngTable *__restrict__ T,
                                                                 const Rng *__restrict__ base, int jb1,
                                                                 const int64_t *__restrict__ order,
                                                                 const int64_t *__restrict__ kfirst,
                                                                 const double *__restrict__ red2, int buckets,
                                                                 const int32_t *__restrict__ uneven,
                                                                 uint64_t *__restrict__ split)
{
    if (kg_.bid == 1) {
        if (*uneven) step_splits(f.rnew, s->n_max, buckets, split);
        return;
    }
    __shared__ double part[ORB_THREADS][NRED];
    __shared__ double acc[NRED];
    const int t = threadIdx.x;
    if (t < NRED) {
        double a = red2[t];
        for (int b = 1; b < RED2_BLOCKS; b++) {
            const double p = red2[RED_STRIDE * b + t];
            a = red_is_max(t) ? (a >= p ? a : p) : a + p;
        }
        acc[t] = a;
    }
    const int64_t nd = deferred(s, P);
    const int64_t n = s->n_max;
    for (int64_t c0 = 0; c0 < nd; c0 += ORB_THREADS) {          // block-uniform
        const int64_t d = c0 + t;
        if (d < nd) {
            const int64_t j = order[d] >> DEFER_SLOT_BITS;
            const double rj = f.r[j], mj = f.m[j];
            const double Ej = f.E[j], J = f.J[j];
            const double E = Ej + phi_s_own(rj, mj, P.inv_nstar, rj);
            int64_t kt = kfirst[order[d] & ((1ll << DEFER_SLOT_BITS) - 1)];
            if (kt >= n) kt = -1;                      // cmc_orbit.c:52-56: circular
            double red[NRED];
            for (int i = 0; i < NRED; i++) red[i] = 0.0;
            int flags = CMCG_SF_LINSCAN, ntry = 0, hits = 0, misses = 0;
            sample_star(SplitNodes{f.r, f.phi}, f, s, P, rng_jump(T, base[1], (uint64_t)j << 20, 20, jb1), n, j,
                        rj, mj, E, Ej, J, kt, flags, ntry, hits, misses, red);
            f.flags[j] = flags;
            f.ntry[j] = ntry;
            count_star(red, flags, ntry, hits, misses);
            for (int i = 0; i < NRED; i++) part[t][i] = red[i];
        }
        __syncthreads();
        if (t < NRED) {
            const int cnt = nd - c0 < ORB_THREADS ? (int)(nd - c0) : ORB_THREADS;
            double a = acc[t];
            for (int u = 0; u < cnt; u++) {
                const double p = part[u][t];
                a = red_is_max(t) ? (a >= p ? a : p) : a + p;
            }
            acc[t] = a;
        }
        __syncthreads();
    }
    __syncthreads();
    if (t == 0) {                           // new_orbits_calculate's results
        s->max_r = acc[0];
        s->Eescaped += acc[1];
        s->Jescaped += acc[2];
        s->TidalMassLoss += acc[3];
        s->Etidal += acc[4];
        s->TidalMassLoss += s->TidalMassLoss_old;    // cmc_utils.c:2210
        s->n_circular = (int64_t)acc[5];
        s->n_removed_E = (int64_t)acc[6];
        s->n_removed_rt = (int64_t)acc[7];
        s->n_destroyed = (int64_t)acc[8];
        s->n_brent = (int64_t)acc[9];
        s->n_linscan = (int64_t)acc[10];
        s->tries_total = (int64_t)acc[11];
        s->tries_max = (int64_t)acc[12];
        s->n_bracket_hit = (int64_t)acc[13];
        s->n_bracket_fallback = (int64_t)acc[14];
    }
}
};

// calc_orbit_new of a batch, one array per output (callers copy each straight into their own).
struct apsides_soa_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P, int64_t first, int64_t count,
                                   const double *__restrict__ E, const double *__restrict__ J, ApsidesOut o)
{
    int64_t i = (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (i >= count) return;
    int64_t j = first + i, n = s->n_max;
    OrbitRS r = calc_orbit(f.r, f.phi, n, j, f.r[j], f.m[j], P, E[i], J[i]);
    if (r.err) dev_set_error(s, r.err, j);
    o.rp[i] = r.rp; o.ra[i] = r.ra; o.dQdrp[i] = r.dQdrp; o.dQdra[i] = r.dQdra;
    o.kmin[i] = r.kmin; o.kmax[i] = r.kmax;
    o.circular[i] = r.circular;
}
};

struct fzq_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P, int64_t count, const int64_t *__restrict__ jj,
                           const int64_t *__restrict__ kmin, const int64_t *__restrict__ kmax,
                           const double *__restrict__ E, const double *__restrict__ J, int64_t *__restrict__ out)
{
    int64_t i = (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (i >= count) return;
    int64_t j = jj[i];
    int64_t k = find_zero_Q(f.r, f.phi, f.r[j], f.m[j], P.inv_nstar, kmin[i], kmax[i], E[i], J[i]);
    if (k < 0) dev_set_error(s, CMCG_E_BRACKET, j);
    out[i] = k;
}
};

struct frv_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P, int64_t count, const int64_t *__restrict__ jj,
                           const int64_t *__restrict__ kk, const double *__restrict__ E,
                           const double *__restrict__ J, double *__restrict__ out)
{
    int64_t i = (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (i >= count) return;
    int64_t j = jj[i];
    const RootVr rv = find_root_vr(f.r, f.phi, f.r[j], f.m[j], P.inv_nstar, P.cenma_m * P.madhoc, kk[i], E[i], J[i]);
    out[i] = rv.root;
    if (rv.bad) dev_set_error(s, CMCG_E_BRENT, j);
}
};

struct pred_from_apsides_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, float2 *__restrict__ pred)
{
    const int64_t j = 1 + (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (j > s->n_max) return;
    const double rp = f.r_peri[j], ra = f.r_apo[j];
    pred[j] = make_float2(rp > 0.0 ? (float)log(rp) : 0.f, ra > 0.0 ? (float)log(ra) : 0.f);
}
};

// ------------------------------------------------------------------ radial index
struct ridx_clear_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, uint32_t *__restrict__ t, int64_t count, int32_t *__restrict__ bad)
{
    if (kg_.bid == 0 && threadIdx.x == 0) *bad = 0;
    for (int64_t i = (int64_t)kg_.bid * blockDim.x + threadIdx.x; i < count; i += (int64_t)kg_.nb * blockDim.x)
        t[i] = 0;
}
};

// The packed (r, phi) node table (nodes 0..n+1) and the radial index's marks
// (nodes 0..n), in one pass over r and phi: node k (node 0
// stands for "below every bucket") writes its index at its bucket when it is the
// bucket's last node, and k at every multiple of RIDX_TILE in (bucket(r_k),
// bucket(r_{k+1})] of the tile table.  The index array and *bad must be cleared before; *bad is
// set where the radii do not ascend (the step's sort then does without their order).
struct node_index_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ r, const double *__restrict__ phi, DevScalars *s,
                                  double2 *__restrict__ nodes, uint32_t *__restrict__ t,
                                  uint32_t *__restrict__ tb, int bits, int32_t *bad)
{
    const int64_t n = s->n_max;
    const int64_t k = (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (k > n + 1) return;
    const double rk = r[k];
    nodes[k] = make_double2(rk, phi[k]);
    if (k > n) return;
    const int64_t nb = (int64_t)1 << bits;
    int64_t bk = -1, bn = nb + 1;
    if (n >= 1) {
        RIdx x;
        x.t = t;
        x.nb = 1u << bits;
        x.lo = (uint64_t)__double_as_longlong(r[1]);
        x.shift = ridx_shift(x.lo, (uint64_t)__double_as_longlong(r[n]), bits);
        if (k >= 1) bk = ridx_bucket(x, rk);
        if (k < n) {
            const double rk1 = r[k + 1];
            bn = ridx_bucket(x, rk1);
            if (k >= 1 && !(rk <= rk1)) *bad = 1;
        }
        if (k >= 1 && bn != bk) t[bk] = (uint32_t)k;
    }
    for (int64_t m = (bk + RIDX_TILE) / RIDX_TILE; m * RIDX_TILE <= bn; m++) tb[m] = (uint32_t)k;
}
};

// The LDS samples of the (r, phi) table for a COARSE-sample launch: node
// min(s * stride, n + 1) for s = 0..cs, from the packed nodes.
__device__ void coarse_build(const double2 *__restrict__ nodes, DevScalars *s, int cs, double2 *__restrict__ out, int i)
{
    if (i == 0) {
        // new_orbits_calculate (cmc_utils.c:2198) and the counters of this call
        s->OldTidalMassLoss = s->TidalMassLoss_old;
        s->n_defer = 0;
    }
    if (i > cs) return;
    const int64_t n = s->n_max;
    const int64_t k = (int64_t)i * coarse_stride(n, cs);
    out[i] = nodes[k < n + 1 ? k : n + 1];
}

// t[b] = the largest marked index below b in its tile, or the tile's entry value:
// an exclusive running maximum, in place.  16 buckets per thread (four 16-byte loads),
// the threads' maxima scanned by wave shuffles and the four wave totals through LDS.
// The blocks after the tiles build the sampler's LDS samples.
struct ridx_scan_kernel {
    static constexpr int LB = 256, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, uint32_t *__restrict__ t, const uint32_t *__restrict__ tb,
                                                        int bits, const double2 *__restrict__ nodes, DevScalars *s, int cs,
                                                        double2 *__restrict__ coarse)
{
    __shared__ uint32_t wtot[4];
    const int64_t entries = ridx_entries(bits);
    if (kg_.bid >= ridx_tiles(bits)) {
        coarse_build(nodes, s, cs, coarse, (int)(kg_.bid - ridx_tiles(bits)) * 256 + threadIdx.x);
        return;
    }
    const int64_t i0 = (int64_t)kg_.bid * RIDX_TILE + 16 * threadIdx.x;
    const bool whole = i0 + 16 <= entries;
    uint32_t v[16];
    if (whole) {
        const uint4 *p = reinterpret_cast<const uint4 *>(t + i0);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint4 x = p[q];
            v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int q = 0; q < 16; q++) v[q] = i0 + q < entries ? t[i0 + q] : 0u;
    }
    uint32_t m = 0;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const uint32_t e = v[q];
        v[q] = m;
        m = e > m ? e : m;
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t inc = m;                                   // inclusive max-scan over the wave
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = __shfl_up(inc, d, 64);
        if (lane >= d) inc = o > inc ? o : inc;
    }
    uint32_t ex = __shfl_up(inc, 1, 64);
    if (lane == 0) ex = 0u;
    if (lane == 63) wtot[w] = inc;
    __syncthreads();
    uint32_t start = tb[kg_.bid];
    for (int q = 0; q < w; q++) start = wtot[q] > start ? wtot[q] : start;
    start = ex > start ? ex : start;
#pragma unroll
    for (int q = 0; q < 16; q++) v[q] = v[q] > start ? v[q] : start;
    if (whole) {
        uint4 *p = reinterpret_cast<uint4 *>(t + i0);
#pragma unroll
        for (int q = 0; q < 4; q++) p[q] = make_uint4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
    } else {
#pragma unroll
        for (int q = 0; q < 16; q++)
            if (i0 + q < entries) t[i0 + q] = v[q];
    }
}
};

// Launch shapes of the orbit sampler that the autotuner chooses from: threads per
// block, LDS samples of the (r, phi) table, and the most lanes one star's tries get
// in a round (64: all idle lanes; fewer: less speculative work).  Every variant gives
// the same stars; only the block order of the escape sums differs.
using OrbFn = void (*)(dim3, dim3, hipStream_t, DevFields, DevScalars *, KParams, const JumpTables *,
                       const Rng *, double *, int64_t *, int64_t *, const float2 *, float, const double2 *, const double2 *,
                       const uint32_t *, int);
template <int THREADS, int COARSE, int CAP, int MINB>
void orbits_launch(dim3 g, dim3 b, hipStream_t st, DevFields f, DevScalars *s, KParams P, const JumpTables *jump,
                   const Rng *base, double *partials, int64_t *defer, int64_t *kfirst, const float2 *pred, float margin,
                   const double2 *nodes, const double2 *coarse,
                   const uint32_t *ridx, int ridx_bits)
{
    kl<orbits_kernel<THREADS, COARSE, CAP, MINB>>(g, b, 0, st, f, s, P, jump, base, partials, defer, kfirst, pred, margin, nodes,
                                                  coarse, ridx, ridx_bits);
}
struct OrbVariant { OrbFn fn; int threads, coarse, cap, minb; };
#define ORB_V(T, C, K, M) {orbits_launch<T, C, K, M>, T, C, K, M}
const OrbVariant kOrbVariants[] = {
    // the first is the default: at most four lanes per star waste few tries.  Its bound of five
    // waves per SIMD costs nothing and gains nothing: the allocation without it takes 91 registers
    // for 89, five waves too (N = 4e6 795 us both, 1e6 185 and 180); the tuner tries both.
    // Sampler time, default / with 64 lanes / 128 threads (whose LDS allows fewer waves): N = 4e6
    // 795 / 868 / 972 us, 1e6 192 / 211 / 257, 3e5 60 / 71 / 87, 1e4 33 / 40 / 39.
    ORB_V(256, 1024, 4, 5),  ORB_V(256, 512, 64, 1), ORB_V(256, 2048, 64, 1), ORB_V(128, 1024, 64, 1),
    ORB_V(512, 1024, 64, 1), ORB_V(128, 512, 64, 1), ORB_V(256, 1024, 2, 1),  ORB_V(256, 1024, 4, 1),
    ORB_V(256, 1024, 8, 1),  ORB_V(256, 512, 4, 1),  ORB_V(256, 1024, 64, 1), ORB_V(256, 512, 4, 5),
    ORB_V(256, 1024, 8, 5)};
#undef ORB_V
constexpr int ORB_NVARIANTS = sizeof(kOrbVariants) / sizeof(kOrbVariants[0]);

int bits_needed(uint64_t x)
{
    int b = 0;
    while (b < 64 && (x >> b)) b++;
    return b;
}
} // namespace

hipError_t launch_orbits(const DevFields &f, DevScalars *s, const KParams &P, const RngTable *T,
                         const Scratch &sc, int64_t n_ub, hipStream_t st, const MlpState *mlp,
                         float margin, hipEvent_t ev_a, hipEvent_t ev_b, int variant, bool pred_fixed, bool index_clear)
{
    const OrbVariant &V = kOrbVariants[variant >= 0 && variant < ORB_NVARIANTS ? variant : 0];
    int64_t nblocks = (n_ub + V.threads - 1) / V.threads;
    if (nblocks < 1) nblocks = 1;
    if (nblocks > sc.max_blocks) return hipErrorInvalidValue;
    int jb1 = 20 + bits_needed((uint64_t)n_ub);
    if (V.coarse > ORB_MAX_COARSE) return hipErrorInvalidValue;
    if (hipError_t e = launch_node_index(f, s, sc, n_ub, V.coarse, index_clear, st)) return e;
    const float2 *pred = nullptr;
    if (mlp) {
        if (!sc.pred) return hipErrorInvalidValue;
        if (!pred_fixed)
            if (hipError_t e = launch_mlp_infer_stars(f, s, P, *mlp, sc.pred, n_ub, st)) return e;
        pred = sc.pred;
    }
    if (ev_a) hipEventRecord(ev_a, st);
    V.fn(dim3((unsigned)nblocks), dim3(V.threads), st, f, s, P, sc.jump, (const Rng *)sc.rng_base,
                       sc.partials, sc.defer_list, sc.defer_kfirst, pred, margin,
                       (const double2 *)sc.nodes, (const double2 *)sc.coarse, (const uint32_t *)sc.ridx, sc.ridx_bits);
    if (ev_b) hipEventRecord(ev_b, st);
    const int buckets = sort_shape(n_ub).buckets;
    kl<after_orbits_kernel>(dim3(RED2_BLOCKS + 1 + DEFER_BLOCKS + 1), dim3(DEFER_T), 0, st, f, s, P, (const double *)sc.partials,
                       nblocks, sc.red2, (const int64_t *)sc.defer_list, sc.defer_kfirst, sc.defer_order, buckets,
                       sc.sort_uneven);
    kl<defer_tail_kernel>(dim3(2), dim3(ORB_THREADS), 0, st, f, s, P, T, sc.rng_base, jb1,
                       (const int64_t *)sc.defer_order, (const int64_t *)sc.defer_kfirst, (const double *)sc.red2, buckets,
                       (const int32_t *)sc.sort_uneven, sc.sort_split);
    return hipGetLastError();
}

hipError_t launch_pred_from_apsides(const DevFields &f, DevScalars *s, const Scratch &sc, int64_t n_ub,
                                    hipStream_t st)
{
    if (!sc.pred) return hipErrorInvalidValue;
    if (n_ub > 0)
        kl<pred_from_apsides_kernel>(dim3((unsigned)((n_ub + 255) / 256)), dim3(256), 0, st, f, s,
                           sc.pred);
    return hipGetLastError();
}

hipError_t launch_node_index(const DevFields &f, DevScalars *s, const Scratch &sc, int64_t n_ub, int coarse, bool clear,
                             hipStream_t st)
{
    const int64_t entries = ridx_entries(sc.ridx_bits);
    if (!clear) kl<ridx_clear_kernel>(dim3(512), dim3(256), 0, st, sc.ridx, entries, sc.sort_uneven);
    kl<node_index_kernel>(dim3((unsigned)((n_ub + 2 + 255) / 256)), dim3(256), 0, st, f.r, f.phi, s,
                       (double2 *)sc.nodes, sc.ridx, sc.ridx_tb, sc.ridx_bits, sc.sort_uneven);
    kl<ridx_scan_kernel>(dim3((unsigned)(ridx_tiles(sc.ridx_bits) + (coarse + 256) / 256)), dim3(256), 0, st, sc.ridx,
                       (const uint32_t *)sc.ridx_tb, sc.ridx_bits, (const double2 *)sc.nodes, s, coarse, sc.coarse);
    return hipGetLastError();
}

int orbit_variant_count() { return ORB_NVARIANTS; }
void orbit_variant_shape(int v, int *threads, int *coarse, int *cap, int *minb)
{
    *threads = kOrbVariants[v].threads;
    *coarse = kOrbVariants[v].coarse;
    if (cap) *cap = kOrbVariants[v].cap;
    if (minb) *minb = kOrbVariants[v].minb;
}

hipError_t launch_apsides_soa(const DevFields &f, DevScalars *s, const KParams &P, int64_t first, int64_t count,
                              const double *E, const double *J, const ApsidesOut &o, hipStream_t st)
{
    if (count <= 0) return hipSuccess;
    kl<apsides_soa_kernel>(dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, f, s, P, first,
                       count, E, J, o);
    return hipGetLastError();
}

hipError_t launch_find_root_vr(const DevFields &f, DevScalars *s, const KParams &P, int64_t count,
                               const int64_t *j, const int64_t *k, const double *E, const double *J, double *out,
                               hipStream_t st)
{
    if (count <= 0) return hipSuccess;
    kl<frv_kernel>(dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, f, s, P, count, j, k, E,
                       J, out);
    return hipGetLastError();
}

hipError_t launch_find_zero_Q(const DevFields &f, DevScalars *s, const KParams &P, int64_t count,
                              const int64_t *j, const int64_t *kmin, const int64_t *kmax,
                              const double *E, const double *J, int64_t *out, hipStream_t st)
{
    if (count <= 0) return hipSuccess;
    kl<fzq_kernel>(dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, f, s, P, count, j, kmin,
                       kmax, E, J, out);
    return hipGetLastError();
}
