// a4 two-body relaxation (src/cmc/cmc_dynamics.c:17-542, relaxation branch
// :427-498), a10 relaxation time step (src/cmc/cmc_dynamics_helper.c:2526-2579),
// calc_sigma_r (:2821-2986), calc_timestep (src/cmc/cmc_utils.c:2132-2148) and the
// per-pair / per-star RNG substream bases.
//
// Relaxation is one thread per radially adjacent pair (2p+1, 2p+2): a pure
// streaming map reading r, m, phi, vr, vt of both stars plus r[k-20], r[k+20]
// (cache-served) and writing vr, vt, E, J, Y: 72 B/star of compulsory HBM traffic.
// The scattering angles' sin/cos are correctly rounded double-double evaluations
// (dd_trig.hpp), so the kicks do not depend on the device math library.
#include "kernels.hpp"
#include "dd_trig.hpp"

namespace {
__device__ __forceinline__ double sqr(double x) { return x * x; }
__device__ __forceinline__ double cub(double x) { return x * x * x; }

// cmc_dynamics_helper.c:768-786 calc_n_local
__device__ __forceinline__ double calc_n_local(const double *__restrict__ r, int64_t k, int64_t p, int64_t N_LIMIT)
{
    int64_t kmin = k - p, kmax = k + p;
    if (kmin < 0) { kmin = 0; kmax = 2 * p + 1; }
    else if (kmax > N_LIMIT) { kmax = N_LIMIT; kmin = N_LIMIT - 2 * p - 1; }
    // clusters smaller than 2p+2 stars would index outside [0, N+1] (undefined in
    // the reference as well); clamp to the array
    if (kmax > N_LIMIT + 1) kmax = N_LIMIT + 1;
    if (kmin < 0) kmin = 0;
    return (2.0 * ((double)p)) * 3.0 / (4.0 * CMCG_PI * (cub(r[kmax]) - cub(r[kmin])));
}

// The step's substream bases: base[0] = seeded state advanced by step * 2^72 (the
// step's relaxation pairs), base[1] = base[0] + 2^70 (its orbit slots), base[2] = base[1] +
// 2^20 (orbit slot 1, the sampler's first).  One wave.
constexpr int RB_T = 64;
constexpr int DT_SLOTS = 64;     // the step's time-step minimum: slots of sigma_dt_kernel (<= RB_T)
__device__ __forceinline__ void rng_bases(const JumpLevel *__restrict__ J, DevScalars *s, const Rng *__restrict__ seeded,
                                          Rng *__restrict__ base, int64_t step_override)
{
    const uint64_t step = step_override >= 0 ? (uint64_t)step_override : s->step;
    const Rng a = jump_uniform(J + JL_STEP, JL_STEP_N, rng_uniform(*seeded), step & 0xffffffffffffffull);
    const Rng b = jump_wave(J[JL_PHASE], a, 16);
    const Rng c = jump_wave(J[JL_SLOT], b, 1);
    if (threadIdx.x == 0) {
        base[0] = a;
        base[1] = b;
        base[2] = c;
    }
}
struct rng_bases_kernel {
    static constexpr int LB = RB_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const JumpLevel *__restrict__ J, DevScalars *s,
                                                         const Rng *__restrict__ seeded, Rng *__restrict__ base,
                                                         int64_t step_override)
{
    rng_bases(J, s, seeded, base, step_override);
}
};

// The jump tables from the generator's matrices, a level a block: thread (c, q, v) applies the
// unit's matrix to v at piece q of word c, 63 times.  (Creating a lone context takes 1.13 ms; 1.18
// when they were formed on the host and their 2.9 MB copied, 1.09 without them.)
struct jump_build_kernel {
    static constexpr int LB = 512, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const RngTable *__restrict__ T, JumpTables *__restrict__ J)
{
    const int level = kg_.bid, t = threadIdx.x, c = t >> 7, q = (t >> 4) & 7, v = t & 15;
    int b0, b1 = -1;                               // the unit: matrix power b0, or b0 and b1 together
    if (level < JL_SLOT) {
        b0 = 6 * (level - JL_PAIR);                // 3 64^k = 2^(6k) + 2^(6k + 1)
        b1 = b0 + 1;
    } else if (level < JL_PHASE) {
        b0 = 20 + 6 * (level - JL_SLOT);
    } else {
        b0 = level == JL_PHASE ? 66 : 72 + 6 * (level - JL_STEP);
    }
    const bool lanes = jump_over_lanes(level);
    uint32_t *L = J->level[level].t;
    uint32_t x = b0 < 128 ? (uint32_t)v << (4 * q) : 0u;
    for (int d = 0; d < 64; d++) {
        L[jump_index(lanes, c, q, v, d)] = x;
        if (level == JL_SLOT) {                    // d slots and 8 d slots
            if (d < 8) J->orbit.lo.t[c][q][v][d] = x;
            if (d % 8 == 0) J->orbit.hi.t[c][q][v][d / 8] = x;
        }
        if (b1 >= 0) x = gf2_matvec(T->col[b1][c], x);
        if (b0 < 128) x = gf2_matvec(T->col[b0][c], x);
    }
}
};

struct rng_draws_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const RngTable *__restrict__ T, const Rng *__restrict__ base, int phase,
                                 int64_t first, int64_t count, int ndraw, double *__restrict__ out, int jb1)
{
    int64_t i = (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (i >= count) return;
    int64_t idx = first + i;
    Rng st;
    if (phase == 0) st = rng_jump(T, base[0], 3ull * (uint64_t)idx, 0, jb1);
    else st = rng_jump(T, base[1], (uint64_t)idx << 20, 20, jb1);
    for (int d = 0; d < ndraw; d++) out[i * ndraw + d] = rng_dbl(st);
}
};

struct dtrel_init_kernel { static constexpr int LB = 1024, MB = 0; static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s) { s->dtrel = __longlong_as_double(0x7ff0000000000000ll); } };

// simul_relax_new: one thread per window si = 1+p, 1+3p, ... (si < N - p), the
// window sums taken in the reference's order, then an order-independent min: the
// bit patterns of non-negative doubles order like the values, so the wave takes the
// minimum pattern with shuffles and publishes it with one atomicMin.  A block (one
// wave) stages its windows' contiguous range in LDS with coalesced loads, as the
// per-element terms m*madhoc and m*madhoc*(vr^2 + vt^2) (the same roundings as the
// reference's loop); windows of more than SR_LDS elements read global memory.
// SR_T windows at most per block, one per lane of the first wave; all SR_B threads
// stage the block's elements (more loads in flight than one wave issues alone).
constexpr int SR_T = 64, SR_B = 256, SR_LDS = 2560;
struct simul_relax_kernel {
    static constexpr int LB = SR_B, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ r, const double *__restrict__ m,
                                                           const double *__restrict__ vr,
                                                           const double *__restrict__ vt, DevScalars *s, KParams P)
{
    __shared__ double stmp[SR_LDS], sq[SR_LDS];
    const unsigned long long kInf = 0x7ff0000000000000ull;
    unsigned long long mine = kInf;
    const int64_t p = P.avekernel, N = s->n_max, len = 2 * p;
    const bool staged = len <= SR_LDS;
    const int G = staged ? (SR_LDS / len < SR_T ? (int)(SR_LDS / len) : SR_T) : SR_T;   // windows per block
    const int64_t w0 = (int64_t)kg_.bid * G;
    const int64_t e0 = 1 + w0 * len;
    if (staged) {
        for (int64_t q = threadIdx.x; q < G * len; q += SR_B) {
            const int64_t k = e0 + q;
            if (k <= N) {
                const double tmp = m[k] * P.madhoc;
                stmp[q] = tmp;
                sq[q] = tmp * (sqr(vr[k]) + sqr(vt[k]));
            }
        }
        __syncthreads();
    }
    const int64_t w = w0 + threadIdx.x;
    const int64_t si = 1 + p + w * 2 * p;
    if (threadIdx.x < G && si < N - p) {
        const int64_t simin = si - p;
        double Mv2ave = 0.0, Mave = 0.0, M2ave = 0.0;
        if (staged) {
            const int64_t q0 = simin - e0;
            for (int64_t q = q0; q < q0 + len; q++) {
                const double tmp = stmp[q];
                Mv2ave += sq[q];
                Mave += tmp;
                M2ave += sqr(tmp);
            }
        } else {
            for (int64_t k = simin; k < simin + len; k++) {
                double tmp = m[k] * P.madhoc;
                Mv2ave += tmp * (sqr(vr[k]) + sqr(vt[k]));
                Mave += tmp;
                M2ave += sqr(tmp);
            }
        }
        Mv2ave /= (double)(2 * p);
        Mave /= (double)(2 * p);
        M2ave /= (double)(2 * p);
        double sigma = sqrt(Mv2ave / Mave);
        double W = 4.0 * sigma / sqrt(3.0 * CMCG_PI);
        double n_local = calc_n_local(r, si, p, N);
        double dt = sqr(2.0 * P.theta_se_max / CMCG_PI) * (CMCG_PI / 32.0) * cub(W) /
                    (((double)P.n_star) * n_local * (4.0 * M2ave));
        if (dt >= 0.0) mine = (unsigned long long)__double_as_longlong(dt);
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        unsigned long long other = __shfl_xor(mine, o, 64);
        mine = other < mine ? other : mine;
    }
    if (threadIdx.x == 0 && mine != kInf) atomicMin((unsigned long long *)&s->dtrel, mine);   // windows: wave 0 only
}
};

// calc_timestep (cmc_utils.c:2132-2148) and GetTimeStep's fallback (cmc_evolution_thr.c:430-432)
__device__ __forceinline__ void timestep_finalize(DevScalars *s)
{
    double Dt = s->dtrel;
    if (Dt == __longlong_as_double(0x7ff0000000000000ll)) Dt = 0.001;
    if ((s->TidalMassLoss_old - s->OldTidalMassLoss) > 0.01) {
        Dt = s->Prev_Dt * 0.8;
    } else if (Dt > 1.1 * s->Prev_Dt && s->Prev_Dt > 0 && (s->TidalMassLoss - s->OldTidalMassLoss) > 0.02) {
        Dt = s->Prev_Dt * 1.1;
    }
    s->Dt = Dt;
    s->TotalTime += Dt;
}
struct timestep_finalize_kernel { static constexpr int LB = 1024, MB = 0; static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s) { timestep_finalize(s); } };
// Begin of a step (cmc.c:246-258, 278): the per-step resets.
__device__ __forceinline__ void step_begin(DevScalars *s)
{
    s->Eescaped_old = s->Eescaped;
    s->Jescaped_old = s->Jescaped;
    s->TidalMassLoss_old = s->TidalMassLoss;
    s->Etidal_old = s->Etidal;
    s->Eescaped = 0.0; s->Jescaped = 0.0; s->TidalMassLoss = 0.0; s->Etidal = 0.0;
    s->n_max_new = s->n_max;
    s->dtrel = __longlong_as_double(0x7ff0000000000000ll);     // the time step's minimum starts at +inf
}
struct step_begin_kernel { static constexpr int LB = 1024, MB = 0; static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s) { step_begin(s); } };

// Block 0: the begin of the step and the minimum over sigma_dt_kernel's slots, which are reset
// for the next step (when dt_part is given; sigma_dt_kernel touches nothing the begin sets),
// the time step (thread 0) with Prev_Dt for the next one (cmc.c:297: only the time step reads
// it), then the step's RNG substream bases.  The other blocks clear the radial index for the
// orbit phase (its flag of radii out of order: block 0).  (Four launches of 4 to 5 us each that
// had no work of their own.)
constexpr int64_t CLEAR_BLK = RB_T * 16;           // index entries per block
struct timestep_rng_bases_kernel {
    static constexpr int LB = RB_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const JumpLevel *__restrict__ J, DevScalars *s,
                                                                  const Rng *__restrict__ seeded,
                                                                  Rng *__restrict__ base,
                                                                  unsigned long long *__restrict__ dt_part,
                                                                  uint32_t *__restrict__ ridx, int64_t entries,
                                                                  int32_t *__restrict__ bad)
{
    if (kg_.bid > 0) {
        const int64_t b0 = (int64_t)(kg_.bid - 1) * CLEAR_BLK;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int64_t i = b0 + 4 * (q * RB_T + threadIdx.x);
            if (i + 4 <= entries) *reinterpret_cast<uint4 *>(ridx + i) = make_uint4(0, 0, 0, 0);
            else
                for (int64_t k = i; k < entries; k++) ridx[k] = 0;
        }
        return;
    }
    if (dt_part) {
        unsigned long long mine = ~dt_part[threadIdx.x * 16];
        dt_part[threadIdx.x * 16] = 0ull;
        const unsigned long long inf = 0x7ff0000000000000ull;
        mine = mine < inf ? mine : inf;
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            const unsigned long long other = __shfl_xor(mine, o, 64);
            mine = other < mine ? other : mine;
        }
        if (threadIdx.x == 0) {
            step_begin(s);
            s->dtrel = __longlong_as_double((long long)mine);
        }
    }
    if (threadIdx.x == 0) {
        timestep_finalize(s);
        s->Prev_Dt = s->Dt;
        *bad = 0;
    }
    rng_bases(J, s, seeded, base, -1);
}
};

// calc_sigma_r at one rank: sigma over the clamped window [si-p, si+p-1]; the
// reference slides running sums, here each window is summed directly.
// The same window sums with the block's range [first - 2p, last + 2p] staged in
// LDS (every window, including the shifted ones at both ends, lies inside it), in
// the same order and expression as sigma_kernel.
constexpr int SIG_T = 512, SIG_MAXP = 64, SIG_LDS = SIG_T + 4 * SIG_MAXP + 1;   // 12 KB

struct sigma_lds_kernel {
    static constexpr int LB = SIG_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ m, const double *__restrict__ vr,
                                                          const double *__restrict__ vt, double *__restrict__ sigma,
                                                          DevScalars *s, KParams P)
{
    __shared__ double a[SIG_LDS], b[SIG_LDS];
    const int64_t N = s->n_max, p = P.avekernel;
    const int64_t first = 1 + (int64_t)kg_.bid * SIG_T;
    if (first > N) return;
    const int64_t last = first + SIG_T - 1 < N ? first + SIG_T - 1 : N;
    const int64_t lo = first - 2 * p > 1 ? first - 2 * p : 1;
    const int64_t hi = last + 2 * p < N ? last + 2 * p : N;
    for (int64_t k = lo + threadIdx.x; k <= hi; k += SIG_T) {
        double mk = m[k] * P.madhoc;
        a[k - lo] = mk;
        b[k - lo] = mk * (sqr(vr[k]) + sqr(vt[k]));
    }
    __syncthreads();
    const int64_t si = first + threadIdx.x;
    if (si > N) return;
    int64_t simin = si - p, simax = simin + (2 * p - 1);
    if (simin < 1) { simin = 1; simax = simin + (2 * p - 1); }
    else if (simax > N) { simax = N; simin = simax - (2 * p - 1); }
    if (simin < 1) simin = 1;
    if (simax > N) simax = N;
    double Mv2ave = 0.0, Mave = 0.0;
    for (int64_t k = simin; k <= simax; k++) {
        Mv2ave += b[k - lo];
        Mave += a[k - lo];
    }
    sigma[si] = sqrt(Mv2ave / Mave);
}
};

struct sigma_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ m, const double *__restrict__ vr,
                             const double *__restrict__ vt, double *__restrict__ sigma, DevScalars *s, KParams P)
{
    int64_t si = 1 + (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    int64_t N = s->n_max, p = P.avekernel;
    if (si > N) return;
    int64_t simin = si - p, simax = simin + (2 * p - 1);
    if (simin < 1) { simin = 1; simax = simin + (2 * p - 1); }
    else if (simax > N) { simax = N; simin = simax - (2 * p - 1); }
    if (simin < 1) simin = 1;      // N < 2p: keep the window inside the array
    if (simax > N) simax = N;
    double Mv2ave = 0.0, Mave = 0.0;
    for (int64_t k = simin; k <= simax; k++) {
        double mk = m[k] * P.madhoc;
        Mv2ave += mk * (sqr(vr[k]) + sqr(vt[k]));
        Mave += mk;
    }
    sigma[si] = sqrt(Mv2ave / Mave);
}
};

// calc_sigma_r and simul_relax_new in one pass (the step's form): each block stages
// m*madhoc and m*madhoc*(vr^2 + vt^2) for its SD_N stars and 2p on either side (the
// roundings of both references' loops, as sigma_lds_kernel and simul_relax_kernel
// take them), writes sigma of its stars, evaluates the relaxation-time windows that
// start among its stars (window w = [1 + 2pw, 1 + 2p(w+1)), the sums in the
// reference's order) and folds the block's smallest dt into one of DT_SLOTS slots
// (128 bytes apart) as an atomicMax of the complemented bit pattern (non-negative
// doubles order like their patterns; 0 is the identity, so the slots start and are
// left at 0); the one-block time-step kernel takes the minimum over the slots.  Needs
// p <= SIG_MAXP.
// Bound by LDS reads, 80 a star for p = 20, when a thread has one star, and by the launch for
// few stars.  For many (SD_MANY) a thread takes SD_PER = 5 neighbours, whose windows share all
// but SD_PER - 1 elements at either end, and reads each element once (18 a star); an odd number
// keeps the lanes' reads off each other's banks.  Each star's sums are still formed one element
// after another.
template <int SD_T, int SD_PER>
struct sigma_dt_kernel {
    static constexpr int LB = SD_T, MB = 0;
    static constexpr int SD_N = SD_T * SD_PER, SD_LDS = SD_N + 4 * SIG_MAXP + 1;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ r, const double *__restrict__ m,
                                                         const double *__restrict__ vr, const double *__restrict__ vt,
                                                         double *__restrict__ sigma, DevScalars *s, KParams P,
                                                         unsigned long long *__restrict__ dt_part)
{
    __shared__ double a[SD_LDS], b[SD_LDS];
    __shared__ unsigned long long wmin[SD_T / 64];
    const unsigned long long kInf = 0x7ff0000000000000ull;
    const int64_t N = s->n_max, p = P.avekernel, len = 2 * p;
    const int64_t first = 1 + (int64_t)kg_.bid * SD_N;
    const int64_t last = first + SD_N - 1 < N ? first + SD_N - 1 : N;
    const int64_t lo = first - 2 * p > 1 ? first - 2 * p : 1;
    const int64_t hi = last + 2 * p < N ? last + 2 * p : N;
    if (first <= N)
        for (int64_t k = lo + threadIdx.x; k <= hi; k += SD_T) {
            const double mk = m[k] * P.madhoc;
            a[k - lo] = mk;
            b[k - lo] = mk * (sqr(vr[k]) + sqr(vt[k]));
        }
    __syncthreads();
    unsigned long long mine = kInf;
    double sg[SD_PER];
    if (first <= N) {
        const int64_t s0 = first + (int64_t)threadIdx.x * SD_PER;
        double Mv2[SD_PER], M[SD_PER];
#pragma unroll
        for (int u = 0; u < SD_PER; u++) Mv2[u] = M[u] = 0.0;
        if (p >= SD_PER && s0 - p >= 1 && s0 + SD_PER - 1 + p - 1 <= N) {
            // no window of the SD_PER is shifted: star u's is elements u .. u + 2p - 1 from s0 - p
            const double *ea = a + (s0 - p - lo), *eb = b + (s0 - p - lo);
            const int n2 = 2 * (int)p;
#pragma unroll
            for (int k = 0; k < SD_PER - 1; k++)
#pragma unroll
                for (int u = 0; u <= k; u++) { Mv2[u] += eb[k]; M[u] += ea[k]; }
#pragma unroll 4
            for (int k = SD_PER - 1; k < n2; k++) {
                const double x = ea[k], y = eb[k];
#pragma unroll
                for (int u = 0; u < SD_PER; u++) { Mv2[u] += y; M[u] += x; }
            }
#pragma unroll
            for (int k = 0; k < SD_PER - 1; k++)
#pragma unroll
                for (int u = k + 1; u < SD_PER; u++) { Mv2[u] += eb[n2 + k]; M[u] += ea[n2 + k]; }
        } else {
            for (int u = 0; u < SD_PER; u++) {
                const int64_t si = s0 + u;
                if (si > N) break;
                int64_t simin = si - p, simax = simin + (2 * p - 1);
                if (simin < 1) { simin = 1; simax = simin + (2 * p - 1); }
                else if (simax > N) { simax = N; simin = simax - (2 * p - 1); }
                if (simin < 1) simin = 1;
                if (simax > N) simax = N;
                double x = 0.0, y = 0.0;
                for (int64_t k = simin; k <= simax; k++) {
                    y += b[k - lo];
                    x += a[k - lo];
                }
                Mv2[u] = y;
                M[u] = x;
            }
        }
#pragma unroll
        for (int u = 0; u < SD_PER; u++) sg[u] = sqrt(Mv2[u] / M[u]);
        // the windows starting at 1 + 2pw in [first, last]; each lies inside [lo, hi]
        const int64_t w0 = (first - 1 + len - 1) / len;
        for (int64_t w = w0 + threadIdx.x; 1 + w * len <= last; w += SD_T) {
            const int64_t wstart = 1 + w * len, wsi = wstart + p;
            if (wsi >= N - p) break;
            double Mv2ave = 0.0, Mave = 0.0, M2ave = 0.0;
            for (int64_t k = wstart; k < wstart + len; k++) {
                const double tmp = a[k - lo];
                Mv2ave += b[k - lo];
                Mave += tmp;
                M2ave += sqr(tmp);
            }
            Mv2ave /= (double)(2 * p);
            Mave /= (double)(2 * p);
            M2ave /= (double)(2 * p);
            const double sw = sqrt(Mv2ave / Mave);
            const double W = 4.0 * sw / sqrt(3.0 * CMCG_PI);
            const double n_local = calc_n_local(r, wsi, p, N);
            const double dt = sqr(2.0 * P.theta_se_max / CMCG_PI) * (CMCG_PI / 32.0) * cub(W) /
                              (((double)P.n_star) * n_local * (4.0 * M2ave));
            if (dt >= 0.0) {
                const unsigned long long bits = (unsigned long long)__double_as_longlong(dt);
                mine = bits < mine ? bits : mine;
            }
        }
    }
    __syncthreads();                           // the sums are done: sigma leaves through a, coalesced
    if (first <= N)
#pragma unroll
        for (int u = 0; u < SD_PER; u++) a[threadIdx.x * SD_PER + u] = sg[u];
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const unsigned long long other = __shfl_xor(mine, o, 64);
        mine = other < mine ? other : mine;
    }
    if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = mine;
    __syncthreads();
    for (int64_t k = first + threadIdx.x; k <= last; k += SD_T) sigma[k] = a[k - first];
    if (threadIdx.x == 0) {
        for (int q = 1; q < SD_T / 64; q++) mine = wmin[q] < mine ? wmin[q] : mine;
        if (mine != kInf) atomicMax(&dt_part[(kg_.bid % DT_SLOTS) * 16], ~mine);
    }
}
};

// Pair pr draws from offset 3 pr (jump_lanes).
// energy_conservation1 (cmc_utils.c:227-236) for star i from its values after the
// relaxation: vtold, vrold and Uoldrold = phi + MPI_PHI_S(r, i)
__device__ __forceinline__ void ec1_star(DevFields &f, const KParams &P, int64_t i, double r, double m, double phi,
                                         double vr, double vt)
{
    f.vtold[i] = vt;
    f.vrold[i] = vr;
    f.Uoldrold[i] = phi + phi_s_own(r, m, P.inv_nstar, r);
}

// EC1: energy_conservation1 fused into the pass (the step's form; the entry point of
// that name keeps its own kernel).  T: threads per block (an autotuned launch shape;
// pair p is thread p of the grid whatever T is, so results do not depend on it).
template <bool EC1, int T>
struct relax_kernel {
    static constexpr int LB = T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, DevFields f, DevScalars *s, KParams P,
                                                    const Rng *__restrict__ base,
                                                    const JumpLevel *__restrict__ J)
{
    int64_t pr = (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    int64_t N = s->n_max;
    Rng rng = jump_lanes(J + JL_PAIR, JL_PAIR_N, base[0], (uint32_t)(pr >> 6));    // before any lane leaves
    if (EC1 && pr == N / 2 && (N & 1)) {    // the unpaired last star keeps its velocities
        ec1_star(f, P, N, f.r[N], f.m[N], f.phi[N], f.vr[N], f.vt[N]);
        return;
    }
    if (pr >= N / 2) return;            // pairs while si <= N - N%2 - 1 (cmc_dynamics.c:203)
    const int64_t k = 2 * pr + 1, kp = k + 1;
    const double dt = s->Dt;

    // calc_encounter_dyns (cmc_dynamics_helper.c:831-871)
    double Y = rng_dbl(rng);
    f.Y[k] = Y;
    f.Y[kp] = Y;
    double phi = Y * 2.0 * CMCG_PI;
    double vrk = f.vr[k], vtk = f.vt[k], vrkp = f.vr[kp], vtkp = f.vt[kp];
    double v[4], vp[4], w[4], w1[4], w2[4];
    v[1] = vtk; v[2] = 0.0; v[3] = vrk;
    double sphi, cphi;
    ddtrig::sincos(phi, &sphi, &cphi);
    vp[1] = vtkp * cphi;
    vp[2] = vtkp * sphi;
    vp[3] = vrkp;
    for (int j = 1; j <= 3; j++) w[j] = vp[j] - v[j];
    double W = sqrt(sqr(w[1]) + sqr(w[2]) + sqr(w[3]));
    if (W == 0.0) { dev_set_error(s, CMCG_E_WZERO, k); return; }

    double n_local = calc_n_local(f.r, k, P.avekernel, N);
    double mass_k = f.m[k], mass_kp = f.m[kp];
    (void)rng_dbl(rng);                 // P_enc test (cmc_dynamics.c:406); P_enc = 0 here

    double Trel12 = (CMCG_PI / 32.0) * cub(W) / (((double)P.n_star) * n_local * sqr((mass_k + mass_kp) * P.madhoc));
    double beta = (CMCG_PI / 2.0) * sqrt(dt / Trel12);
    if (beta > CMCG_PI / 2.0) beta = CMCG_PI / 2.0;
    double wp = sqrt(sqr(w[1]) + sqr(w[2]));
    if (wp == 0.0) { dev_set_error(s, CMCG_E_WPZERO, k); return; }
    w1[1] = -w[2] * W / wp;
    w1[2] = w[1] * W / wp;
    w1[3] = 0.0;
    w2[1] = -w[1] * w[3] / wp;
    w2[2] = -w[2] * w[3] / wp;
    w2[3] = wp;
    double psi = rng_dbl(rng) * 2 * CMCG_PI;
    double cb, sb, cp, sp;
    ddtrig::sincos(beta, &sb, &cb);
    ddtrig::sincos(psi, &sp, &cp);
    double v_new[4], vp_new[4];
    for (int j = 1; j <= 3; j++) {
        double w_new = w[j] * cb + w1[j] * sb * cp + w2[j] * sb * sp;
        v_new[j] = v[j] - mass_kp / (mass_k + mass_kp) * (w_new - w[j]);
        vp_new[j] = vp[j] + mass_k / (mass_k + mass_kp) * (w_new - w[j]);
    }
    double nvr_k = v_new[3], nvt_k = sqrt(sqr(v_new[1]) + sqr(v_new[2]));
    double nvr_kp = vp_new[3], nvt_kp = sqrt(sqr(vp_new[1]) + sqr(vp_new[2]));
    f.vr[k] = nvr_k; f.vt[k] = nvt_k;
    f.vr[kp] = nvr_kp; f.vt[kp] = nvt_kp;
    // set_star_EJ (cmc_dynamics_helper.c:878-882), old phi and r
    const double phik = f.phi[k], phikp = f.phi[kp], rk = f.r[k], rkp = f.r[kp];
    f.E[k] = phik + 0.5 * (sqr(nvr_k) + sqr(nvt_k));
    f.J[k] = rk * nvt_k;
    f.E[kp] = phikp + 0.5 * (sqr(nvr_kp) + sqr(nvt_kp));
    f.J[kp] = rkp * nvt_kp;
    if (EC1) {
        ec1_star(f, P, k, rk, mass_k, phik, nvr_k, nvt_k);
        ec1_star(f, P, kp, rkp, mass_kp, phikp, nvr_kp, nvt_kp);
    }
}
};

int bits_needed(uint64_t x)
{
    int b = 0;
    while (b < 64 && (x >> b)) b++;
    return b;
}
} // namespace

hipError_t launch_jump_build(const RngTable *T, JumpTables *J, hipStream_t st)
{
    kl<jump_build_kernel>(dim3(JL_COUNT), dim3(512), 0, st, T, J);
    return hipGetLastError();
}

hipError_t launch_rng_bases(DevScalars *s, const Scratch &sc, hipStream_t st)
{
    kl<rng_bases_kernel>(dim3(1), dim3(RB_T), 0, st, (const JumpLevel *)sc.jump->level, s, sc.rng_seeded, sc.rng_base, (int64_t)-1);
    return hipGetLastError();
}

hipError_t launch_rng_bases_step(DevScalars *s, const Scratch &sc, int64_t step, hipStream_t st)
{
    kl<rng_bases_kernel>(dim3(1), dim3(RB_T), 0, st, (const JumpLevel *)sc.jump->level, s, sc.rng_seeded, sc.rng_base, step);
    return hipGetLastError();
}

// Packed (r, phi) nodes for the searches and the middle table (every MID_STEP-th node).
struct mid_build_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ r, const double *__restrict__ phi, DevScalars *s,
                                 double2 *__restrict__ nodes, double2 *__restrict__ mid)
{
    int64_t k = (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (k > s->n_max + 1) return;
    double2 v = make_double2(r[k], phi[k]);
    nodes[k] = v;
    if (k % MID_STEP == 0) mid[k / MID_STEP] = v;
}
};

hipError_t launch_mid_build(const DevFields &f, DevScalars *s, const Scratch &sc, int64_t n_ub, hipStream_t st)
{
    int64_t nn = n_ub + 2;
    kl<mid_build_kernel>(dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, st, f.r, f.phi, s,
                       sc.nodes, sc.mid);
    return hipGetLastError();
}

hipError_t launch_rng_draws(const RngTable *T, const Rng *base, int phase, int64_t first, int64_t count,
                            int ndraw, double *out, hipStream_t st)
{
    if (count <= 0) return hipSuccess;
    uint64_t last = (uint64_t)(first + count);
    int jb1 = phase == 0 ? bits_needed(3ull * last) : 20 + bits_needed(last);
    kl<rng_draws_kernel>(dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, T, base, phase,
                       first, count, ndraw, out, jb1);
    return hipGetLastError();
}

hipError_t launch_sigma(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, hipStream_t st)
{
    if (n_ub <= 0) return hipSuccess;
    if (P.avekernel <= SIG_MAXP)
        kl<sigma_lds_kernel>(dim3((unsigned)((n_ub + SIG_T - 1) / SIG_T)), dim3(SIG_T), 0, st, f.m,
                           f.vr, f.vt, f.sigma, s, P);
    else
        kl<sigma_kernel>(dim3((unsigned)((n_ub + 255) / 256)), dim3(256), 0, st, f.m, f.vr, f.vt,
                           f.sigma, s, P);
    return hipGetLastError();
}

hipError_t launch_simul_relax(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, hipStream_t st,
                              bool init_min)
{
    if (init_min) kl<dtrel_init_kernel>(dim3(1), dim3(1), 0, st, s);
    const int64_t nw = n_ub / (2 * P.avekernel) + 1;
    const int64_t len = 2 * P.avekernel;
    const int64_t G = len <= SR_LDS ? (SR_LDS / len < SR_T ? SR_LDS / len : SR_T) : SR_T;   // as in the kernel
    kl<simul_relax_kernel>(dim3((unsigned)((nw + G - 1) / G)), dim3(SR_B), 0, st, f.r, f.m, f.vr,
                       f.vt, s, P);
    return hipGetLastError();
}

template <int T, int PER>
void sigma_dt_launch(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc, int64_t n_ub, hipStream_t st)
{
    kl<sigma_dt_kernel<T, PER>>(dim3((unsigned)((n_ub + T * PER - 1) / (T * PER))), dim3(T), 0, st, f.r, f.m, f.vr, f.vt,
                                f.sigma, s, P, sc.dt_part);
}
// One star a thread fills the chip from fewer stars: 12 / 17 us at 3e5 (one / five a thread),
// 24 / 24 at 1e6, 41 / 33 at 2e6, 72 / 48 at 4e6.
constexpr int64_t SD_MANY = 1500000;

// The step's begin and time-step phase: calc_sigma_r and simul_relax_new in one pass (or, for
// a window longer than the pass stages, their own kernels), then Dt, the RNG bases and the
// cleared radial index of the orbit phase.
hipError_t launch_timestep_sigma(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc,
                                 int64_t n_ub, hipStream_t st)
{
    const bool one_pass = P.avekernel <= SIG_MAXP && n_ub > 0;
    if (one_pass) {
        if (n_ub > SD_MANY) sigma_dt_launch<128, 5>(f, s, P, sc, n_ub, st);
        else sigma_dt_launch<512, 1>(f, s, P, sc, n_ub, st);
    } else {
        kl<step_begin_kernel>(dim3(1), dim3(1), 0, st, s);
        if (hipError_t e = launch_simul_relax(f, s, P, n_ub, st, false)) return e;
        if (hipError_t e = launch_sigma(f, s, P, n_ub, st)) return e;
    }
    const int64_t entries = ridx_entries(sc.ridx_bits);
    kl<timestep_rng_bases_kernel>(dim3(1 + (unsigned)((entries + CLEAR_BLK - 1) / CLEAR_BLK)), dim3(RB_T), 0, st,
                       (const JumpLevel *)sc.jump->level, s, sc.rng_seeded, sc.rng_base,
                       one_pass ? sc.dt_part : (unsigned long long *)nullptr, sc.ridx, entries, sc.sort_uneven);
    return hipGetLastError();
}
hipError_t launch_timestep_finalize(DevScalars *s, hipStream_t st)
{
    kl<timestep_finalize_kernel>(dim3(1), dim3(1), 0, st, s);
    return hipGetLastError();
}

template <bool EC1, int TH>
void relax_launch(int64_t nth, hipStream_t st, const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc)
{
    kl<relax_kernel<EC1, TH>>(dim3((unsigned)((nth + TH - 1) / TH)), dim3(TH), 0, st, f, s, P,
                              (const Rng *)sc.rng_base, (const JumpLevel *)sc.jump->level);
}

template <bool EC1>
hipError_t relax_launch_shape(int threads, int64_t nth, hipStream_t st, const DevFields &f, DevScalars *s,
                              const KParams &P, const Scratch &sc)
{
    switch (threads) {
    case 128: relax_launch<EC1, 128>(nth, st, f, s, P, sc); break;
    case 256: relax_launch<EC1, 256>(nth, st, f, s, P, sc); break;
    case 512: relax_launch<EC1, 512>(nth, st, f, s, P, sc); break;
    case 1024: relax_launch<EC1, 1024>(nth, st, f, s, P, sc); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_relax(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc,
                        int64_t n_ub, hipStream_t st, bool with_ec1, int threads)
{
    int64_t npairs = n_ub / 2;
    if (with_ec1) {
        // one thread more for an unpaired last star
        const int64_t nth = (n_ub + 1) / 2;
        if (nth <= 0) return hipSuccess;
        return relax_launch_shape<true>(threads, nth, st, f, s, P, sc);
    }
    if (npairs <= 0) return hipSuccess;
    return relax_launch_shape<false>(threads, npairs, st, f, s, P, sc);
}
