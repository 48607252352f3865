// Internal declarations of the cmcg HIP library (gfx950).
//
// Device data layout (all in HBM, one allocation per field, SoA):
//   r, m, phi           : N+2 doubles, the reference's star_r/star_m/star_phi with
//                         sentinels at 0 and N+1 (src/cmc/cmc_utils.c:713-714,
//                         src/cmc/cmc_fits.c:128-129)
//   vr, vt, E, J, ...   : per-star fields at slots 1..N (the AoS star_t fields the
//                         path touches, include/cmc/cmc.h:409-601)
// Every double expression below is written in the reference's operand order and the
// library is compiled with -ffp-contract=off, so the results equal the CPU
// reference's on the same inputs (except libm sin/cos, ~1 ulp).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include "../../include/cmcg.h"
#include "seg.hpp"

#define CMCG_SF_INFINITY 1.0e10
#define CMCG_ZERO 1.0e-20
#define CMCG_PI 3.14159265358979323
#define CMCG_N_TRY 50000

// ---------------------------------------------------------------- device scalars
// Lives in device memory so that a whole step can run without host round trips.
struct DevScalars {
    int64_t n_max, n_max_new;
    double Mtotal, Rtidal, max_r, Dt, Prev_Dt, TotalTime;
    double TidalMassLoss, TidalMassLoss_old, OldTidalMassLoss;
    double Eescaped, Jescaped, Etidal, Eoops;
    double Etot, Ekin, Epot;
    uint64_t step;
    double Eescaped_old, Jescaped_old, Etidal_old;
    // per-call work
    double DTidalMassLoss;
    int32_t error; int32_t pad0;
    int64_t error_index;
    int64_t reserved0;
    int64_t n_excess;            // set_velocities3 stars with vnew2 <= 0
    int64_t first_inf;           // potential_calculate: first slot with r >= SF_INFINITY
    int64_t n_defer;             // orbit phase: stars whose own-index Q <= 0 (linear-scan path)
    int64_t sort_n;              // sort: live stars after dropping the r == SF_INFINITY tail
    int64_t sort_in;             // sort: slots sorted (N_MAX_NEW before the sort)
    // orbit statistics
    int64_t n_circular, n_removed_E, n_removed_rt, n_destroyed, n_brent, n_linscan;
    int64_t tries_total, tries_max, n_bracket_hit, n_bracket_fallback;
    double dtrel;
};

// RNG jump table: g_pow[b][j][i] = column i of T_j^(2^b), b < 128.
struct RngTable { uint32_t col[128][4][32]; };

struct Rng { uint32_t z0, z1, z2, z3; };

// ---------------------------------------------------------------- device fields
struct DevFields {
    double *r, *m, *phi;
    double *vr, *vt, *E, *J;
    int64_t *id;
    double *rnew, *vrnew, *vtnew, *X, *Y, *r_peri, *r_apo;
    double *rOld, *Uoldrold, *Uoldrnew, *vrold, *vtold, *EI;
    double *sigma, *pot_rnew;
    int32_t *ntry, *flags;
    int32_t *knew;         // orbit phase: largest k with r_k < rnew among the old nodes, -1 for a star that leaves
};

struct KParams {
    int64_t n_star;
    double inv_nstar;      // 1.0/N_STAR exactly as the reference's (1.0/clus.N_STAR)
    double madhoc;         // 1.0/((double)N_STAR), cmc_utils.c:1183
    double cenma_m;
    double orbit_r;
    double theta_se_max;
    double gamma;
    int64_t avekernel;
    int32_t chain_k_drop;  // test hook: potential chains' error bound widened by 2^chain_k_drop
    int32_t pad0;
    int64_t defer_cap;     // capacity of the deferred-star list: a power of two above the star capacity
};

__device__ __forceinline__ void dev_set_error(DevScalars *s, int code, int64_t idx)
{
    if (atomicCAS(&s->error, 0, code) == 0) s->error_index = idx;
}

// ---------------------------------------------------------------- taus113
// One step of src/libs/taus113-v2.c:166-177 (32-bit arithmetic replaces the MASK).
__device__ __forceinline__ uint32_t rng_int(Rng &s)
{
    uint32_t b;
    b = ((s.z0 << 6) ^ s.z0) >> 13;  s.z0 = ((s.z0 & 4294967294u) << 18) ^ b;
    b = ((s.z1 << 2) ^ s.z1) >> 27;  s.z1 = ((s.z1 & 4294967288u) << 2) ^ b;
    b = ((s.z2 << 13) ^ s.z2) >> 21; s.z2 = ((s.z2 & 4294967280u) << 7) ^ b;
    b = ((s.z3 << 3) ^ s.z3) >> 12;  s.z3 = ((s.z3 & 4294967168u) << 13) ^ b;
    return s.z0 ^ s.z1 ^ s.z2 ^ s.z3;
}
// taus113-v2.c:187-189
__device__ __forceinline__ double rng_dbl(Rng &s) { return (double)rng_int(s) / 4294967296.0; }

__device__ __forceinline__ uint32_t gf2_matvec(const uint32_t *__restrict__ col, uint32_t v)
{
    uint32_t out = 0;
#pragma unroll
    for (int i = 0; i < 32; i++) out ^= col[i] & (0u - ((v >> i) & 1u));
    return out;
}

// Jump the state forward by `off` steps, using bits [b0, b1) of `off` (the caller
// knows the rest are zero).  Loops are uniform over bit positions, so the matrix
// columns are wave-uniform loads.
__device__ __forceinline__ Rng rng_jump(const RngTable *__restrict__ T, Rng s, uint64_t off, int b0, int b1)
{
    for (int b = b0; b < b1; b++) {
        if (!((off >> b) & 1ull)) continue;
        s.z0 = gf2_matvec(T->col[b][0], s.z0);
        s.z1 = gf2_matvec(T->col[b][1], s.z1);
        s.z2 = gf2_matvec(T->col[b][2], s.z2);
        s.z3 = gf2_matvec(T->col[b][3], s.z3);
    }
    return s;
}

// Jumps of a wave-uniform state.  Level L of the jump tables holds, for d = 0..63, the
// GF(2) matrix of d U_L steps (U_L the level's unit), stored as its products with the 16
// values v of every 4-bit piece q of state word c.  Over the lanes, d = lane, the tables
// are t[c][q][v][d]: a jump is 32 coalesced loads and XORs, and no lookup waits on another
// (through per-block LDS tables of single powers a lane's jump took six to eight dependent
// rounds of 32 lookups: 192 to 256 LDS reads and about 1000 vector instructions a wave).
// Offsets beyond 63 units take the next levels' digits (units grow by 64), the same for the
// whole wave; those levels are t[d][c][q][v], 2 KB a digit.
struct JumpLevel { uint32_t t[4 * 8 * 16 * 64]; };
constexpr int JL_PAIR = 0, JL_PAIR_N = 6;       // units 3 64^k: relaxation pairs (k = 0 over the lanes)
constexpr int JL_SLOT = 6, JL_SLOT_N = 6;       // units 2^20 64^k: orbit slots
constexpr int JL_PHASE = 12;                    // unit 2^66: 16 of them from the pairs to the slots of a step
constexpr int JL_STEP = 13, JL_STEP_N = 10;     // units 2^72 64^k: steps
constexpr int JL_COUNT = JL_STEP + JL_STEP_N;
__host__ __device__ constexpr bool jump_over_lanes(int level) { return level == JL_PAIR; }
__host__ __device__ constexpr int jump_index(bool lanes, int c, int q, int v, int d)
{
    return lanes ? ((c * 8 + q) * 16 + v) * 64 + d : ((d * 4 + c) * 8 + q) * 16 + v;
}

// `lane` steps of the unit of a level over the lanes, from z (uniform over the wave)
__device__ __forceinline__ Rng jump_digit(const JumpLevel &L, const Rng &z, uint32_t lane)
{
    auto word = [&](int c, uint32_t x) {
        uint32_t o = 0;
#pragma unroll
        for (int q = 0; q < 8; q++) o ^= L.t[jump_index(true, c, q, (x >> (4 * q)) & 15u, lane)];
        return o;
    };
    return Rng{word(0, z.z0), word(1, z.z1), word(2, z.z2), word(3, z.z3)};
}
__device__ __forceinline__ Rng rng_uniform(const Rng &z)
{
    auto u = [](uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); };
    return Rng{u(z.z0), u(z.z1), u(z.z2), u(z.z3)};
}
// A uniform jump by a whole wave (every lane active): lane 8 c + q looks up piece q of
// word c, so it is one load and a XOR over eight lanes.  (As 32 scalar loads the compiler
// waits for nearly each: 8 us a jump from cold caches.)
__device__ __forceinline__ Rng jump_wave(const JumpLevel &L, const Rng &z, uint32_t d)
{
    const int i = threadIdx.x & 31, c = i >> 3, q = i & 7;
    const uint32_t zc = c == 0 ? z.z0 : c == 1 ? z.z1 : c == 2 ? z.z2 : z.z3;
    uint32_t o = L.t[jump_index(false, c, q, (zc >> (4 * q)) & 15u, d)];
#pragma unroll
    for (int m = 1; m < 8; m <<= 1) o ^= (uint32_t)__shfl_xor((int)o, m, 64);
    auto word = [&](int lane) { return (uint32_t)__builtin_amdgcn_readlane((int)o, lane); };
    return Rng{word(0), word(8), word(16), word(24)};
}
// the same for an offset w (uniform) of any number of digits
__device__ __forceinline__ Rng jump_uniform(const JumpLevel *__restrict__ L, int levels, Rng z, uint64_t w)
{
    for (int k = 0; k < levels && w; k++, w >>= 6) {
        const uint32_t d = (uint32_t)w & 63u;
        if (d) z = jump_wave(L[k], z, d);
    }
    return z;
}
// The orbit sampler's lanes jump through LDS instead, in two digits of 8, lane = 8 h + l: the
// products for h 8 units are looked up by the wave together (lane 8 h + q takes piece q of
// each word), those for l by each lane in LDS, 32 lookups.  t[c][q][v][d]: the product of
// d U (d 8 U) with value v of piece q of word c.  (Lane tables as above evict the sampler's
// nodes from the L1: 1071 -> 1172 us at N = 4e6; as a pass before it they took 58 us; single
// powers of two, 192 LDS lookups, took about 700 of its 5700 vector instructions a wave.)
struct LaneDigit { uint32_t t[4][8][16][8]; };
struct LaneDigits { LaneDigit lo, hi; };
__device__ __forceinline__ uint32_t xor_over_8_lanes(uint32_t x)
{
    x ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xB1, 0xf, 0xf, true);      // quad_perm [1, 0, 3, 2]
    x ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x4E, 0xf, 0xf, true);      // quad_perm [2, 3, 0, 1]
    x ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x141, 0xf, 0xf, true);     // row_half_mirror
    return x;
}
// z uniform over the wave, every lane active; lo in LDS
__device__ __forceinline__ Rng jump_lane_digits(const LaneDigit &hi, const LaneDigit &lo, const Rng &z)
{
    const int lane = threadIdx.x & 63, g = lane >> 3, l = lane & 7;
    auto upper = [&](int c, uint32_t x) { return xor_over_8_lanes(hi.t[c][l][(x >> (4 * l)) & 15u][g]); };
    const Rng s{upper(0, z.z0), upper(1, z.z1), upper(2, z.z2), upper(3, z.z3)};
    auto lower = [&](int c, uint32_t x) {
        uint32_t o = 0;
#pragma unroll
        for (int q = 0; q < 8; q++) o ^= lo.t[c][q][(x >> (4 * q)) & 15u][l];
        return o;
    };
    return Rng{lower(0, s.z0), lower(1, s.z1), lower(2, s.z2), lower(3, s.z3)};
}
// what a device holds of them
struct JumpTables {
    JumpLevel level[JL_COUNT];
    LaneDigits orbit;
};

// The state of the lane's pair: the wave's first is number 64 w after base.  Every lane of
// the wave calls it.
__device__ __forceinline__ Rng jump_lanes(const JumpLevel *__restrict__ L, int levels, const Rng &base, uint32_t w)
{
    const Rng z = jump_uniform(L + 1, levels - 1, rng_uniform(base), (uint32_t)__builtin_amdgcn_readfirstlane((int)w));
    return jump_digit(L[0], z, threadIdx.x & 63u);
}

// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.  This
// bijection gives XCD x a contiguous range of logical blocks, so the blocks that
// share an L2 work on neighbouring stars and their search paths overlap.
__device__ __forceinline__ int64_t xcd_block(const KGrid &kg)
{
    const int64_t nb = kg.nb, b = kg.bid;
    const int64_t x = b & 7, local = b >> 3, q = nb >> 3, rem = nb & 7;
    return x * q + (x < rem ? x : rem) + local;
}

// ---------------------------------------------------------------- potential helpers
// include/cmc/cmc.h:2175 MPI_PHI_S(rad, j)
__device__ __forceinline__ double phi_s(const double *__restrict__ r, const double *__restrict__ m,
                                        double inv_nstar, double rad, int64_t j)
{
    return (rad >= r[j] ? m[j] / rad : m[j] / r[j]) * inv_nstar;
}
__device__ __forceinline__ double phi_s_own(double rj, double mj, double inv_nstar, double rad)
{
    return mj / (rad >= rj ? rad : rj) * inv_nstar;
}

// cmc_utils.c:1654-1662 function_q evaluated in double (the reference uses x87
// long double here; the oracle measures how often the sign differs).
__device__ __forceinline__ double function_q(double rj, double mj, double inv_nstar,
                                             double r, double pot, double E, double J)
{
    double Jor = J / r;
    double Jr = Jor * Jor;
    double phis = (r >= rj ? mj / r : mj / rj) * inv_nstar;
    return 2.0 * (E - (pot + phis)) - Jr;
}

// What the sign of a star's function_q needs at every node: s0 = (m_j / r_j) / N and
// s1 = m_j / N, the star's own term below and (times 1 / r) above its radius.
struct QStar {
    double rj, mj, inv, E, J;
    double s0, s1, J2, c1, k;
};
__device__ __forceinline__ QStar q_star(double rj, double mj, double inv_nstar, double E, double J)
{
    QStar q;
    q.rj = rj; q.mj = mj; q.inv = inv_nstar; q.E = E; q.J = J;
    q.s0 = mj / rj * inv_nstar;
    q.s1 = mj * inv_nstar;
    q.J2 = J * J;
    q.c1 = __builtin_fabs(E) + __builtin_fabs(q.s0);
    q.k = __builtin_fma(0x1p-42, q.J2, 1e-290);
    return q;
}

// Sign of function_q(rj, mj, inv_nstar, r, pot, E, J) as that function computes it in
// double: -1 (Q < 0), 0 (Q == 0), 1 (Q > 0), 2 (NaN).  Without a division: g = Q r^2 =
// 2 ((E - pot) r - s) r - J^2, s = s0 r below r_j and s1 above, and each of g and the
// computed Q r^2 differs from the exact value by less than 10 2^-53 S r^2, S = 2 (|E| +
// |pot| + |s0|) + (J / r)^2, since each evaluation rounds at most ten times; when |g| exceeds
// 2^-42 S r^2 (plus 1e-290, for products that underflow) the signs agree, otherwise
// function_q itself decides.  (With the reciprocal of r by two Newton steps, as before, a
// sign took about 45 vector instructions, now 20; the samples' two bisections alone take 20 signs.)
__device__ __forceinline__ int q_sign(const QStar &q, double r, double pot)
{
    const double t = q.E - pot, r2 = r + r;
    const double s = r >= q.rj ? q.s1 : q.s0 * r;
    const double g = __builtin_fma(__builtin_fma(t, r, -s), r2, -q.J2);
    const double thr = __builtin_fma((q.c1 + __builtin_fabs(pot)) * r, r2 * 0x1p-42, q.k);
    if (__builtin_fabs(g) > thr) return g < 0.0 ? -1 : 1;
    const double qe = function_q(q.rj, q.mj, q.inv, r, pot, q.E, q.J);
    return qe < 0.0 ? -1 : (qe > 0.0 ? 1 : (qe == 0.0 ? 0 : 2));
}
__device__ __forceinline__ bool q_lt0(int sg) { return sg == -1; }
__device__ __forceinline__ bool q_gt0(int sg) { return sg == 1; }
__device__ __forceinline__ bool q_ge0(int sg) { return sg == 0 || sg == 1; }
__device__ __forceinline__ bool q_le0(int sg) { return sg == -1 || sg == 0; }

// Access to the (r, phi) nodes: the two global arrays, or a packed copy of 16-byte
// (r, phi) nodes, whose Q evaluations and interpolations touch one cache line per
// node instead of two.  Both hold the same values.
struct SplitNodes {
    const double *__restrict__ r;
    const double *__restrict__ phi;
    __device__ __forceinline__ double R(int64_t k) const { return r[k]; }
    __device__ __forceinline__ double P(int64_t k) const { return phi[k]; }
    __device__ __forceinline__ void RP(int64_t k, double &a, double &b) const { a = r[k]; b = phi[k]; }
};
struct PackedNodes {
    const double2 *__restrict__ rp;
    __device__ __forceinline__ double R(int64_t k) const { return rp[k].x; }
    __device__ __forceinline__ double P(int64_t k) const { return rp[k].y; }
    __device__ __forceinline__ void RP(int64_t k, double &a, double &b) const
    {
        double2 v = rp[k];
        a = v.x;
        b = v.y;
    }
};

// cmc_nr.c:62-82 FindZero_r: largest k in [kmin, kmax] with r[k] < x (for sorted r).
template <class N>
__device__ __forceinline__ int64_t find_zero_r_n(const N &nd, int64_t kmin, int64_t kmax, double x)
{
    int guard = 0;
    do {
        int64_t ktry = (kmin + kmax + 1) / 2;
        if (nd.R(ktry) < x) kmin = ktry;
        else kmax = ktry - 1;
    } while (kmax != kmin && ++guard < 96);
    return kmin;
}
__device__ __forceinline__ int64_t find_zero_r(const double *__restrict__ r, int64_t kmin, int64_t kmax, double x)
{
    return find_zero_r_n(SplitNodes{r, nullptr}, kmin, kmax, x);
}

// cmc_utils.c:112-165 potential(r); the bisection bracket [lo, hi] may be narrowed
// by the caller to any [lo, hi] with r[lo] < x <= r[hi] (lo >= 1): the result is the
// unique largest k with r[k] < x, identical to the full-range search.
template <class N>
__device__ __forceinline__ double potential_at_n(const N &nd, int64_t n_max, double x, int64_t lo, int64_t hi,
                                                 bool *bad, int32_t *k_out = nullptr)
{
    if (k_out) *k_out = 0;
    if (x == 0.0) return nd.P(0);
    double r1 = nd.R(1);
    if (x < r1) {
        double p0 = nd.P(0);
        return p0 - (p0 - nd.P(1)) * r1 / x;
    }
    int64_t i;
    if (lo == hi - 1) i = lo;
    else i = find_zero_r_n(nd, lo, hi, x);
    if (i > n_max) { *bad = true; return 0.0; }   // x beyond the outer sentinel
    if (k_out) *k_out = (int32_t)i;
    double ri, pi, ri1, pi1;
    nd.RP(i, ri, pi);
    nd.RP(i + 1, ri1, pi1);
    if (ri > x || ri1 < x) { *bad = true; return 0.0; }
    if (i == 0) return pi1;
    return pi + (pi1 - pi) * (1.0 / ri - 1.0 / x) / (1.0 / ri - 1.0 / ri1);
}
__device__ __forceinline__ double potential_at(const double *__restrict__ r, const double *__restrict__ phi,
                                               int64_t n_max, double x, int64_t lo, int64_t hi, bool *bad)
{
    return potential_at_n(SplitNodes{r, phi}, n_max, x, lo, hi, bad);
}

// cmc_nr.c:316-383 find_zero_Q.  Returns -1 if the bracket cannot close.
template <class N>
__device__ __forceinline__ int64_t find_zero_Q_n(const N &nd, double rj, double mj, double inv_nstar,
                                                 int64_t kmin, int64_t kmax, double E, double J)
{
    const QStar q = q_star(rj, mj, inv_nstar, E, J);
    double a, b, a2, b2;
    nd.RP(kmin, a, b);
    nd.RP(kmax, a2, b2);
    // the direction test qmin < qmax: decided by the signs when they differ
    const int smin = q_sign(q, a, b), smax = q_sign(q, a2, b2);
    bool up;
    if ((smin == -1 || smin == 1) && (smax == -1 || smax == 1) && smin != smax) up = smin < smax;
    else up = function_q(rj, mj, inv_nstar, a, b, E, J) < function_q(rj, mj, inv_nstar, a2, b2, E, J);
    int guard = 0;
    if (up) {
        do {
            int64_t ktry = (kmin + kmax + 1) / 2;
            nd.RP(ktry, a, b);
            if (q_lt0(q_sign(q, a, b))) kmin = ktry;
            else kmax = ktry - 1;
        } while (kmax != kmin && ++guard < 96);
    } else {
        do {
            int64_t ktry = (kmin + kmax + 1) / 2;
            nd.RP(ktry, a, b);
            if (q_gt0(q_sign(q, a, b))) kmin = ktry;
            else kmax = ktry - 1;
        } while (kmax != kmin && ++guard < 96);
    }
    return guard >= 96 ? -1 : kmin;
}
__device__ __forceinline__ int64_t find_zero_Q(const double *__restrict__ r, const double *__restrict__ phi,
                                               double rj, double mj, double inv_nstar,
                                               int64_t kmin, int64_t kmax, double E, double J)
{
    return find_zero_Q_n(SplitNodes{r, phi}, rj, mj, inv_nstar, kmin, kmax, E, J);
}

// cmc_orbit.c:722-740 set_a_b, from the interval's two nodes (k > 0)
__device__ __forceinline__ void set_a_b_nodes(double rj, double mj, const KParams &P, double rk, double pk, double rk1,
                                              double pk1, double *a, double *b)
{
    double Uk = pk + phi_s_own(rj, mj, P.inv_nstar, rk);
    double Uk1 = pk1 + phi_s_own(rj, mj, P.inv_nstar, rk1);
    *a = (Uk1 - Uk) / (1. / rk1 - 1. / rk);
    *b = (Uk / rk1 - Uk1 / rk) / (1. / rk1 - 1. / rk);
}
template <class N>
__device__ __forceinline__ void set_a_b_n(const N &nd, double rj, double mj, const KParams &P, int64_t k,
                                          double *a, double *b)
{
    if (k == 0) {
        double r1, p1;
        nd.RP(1, r1, p1);
        *a = -P.cenma_m * P.madhoc;
        *b = p1 + P.cenma_m * P.madhoc / r1 + mj * P.madhoc / rj;
    } else {
        double rk, pk, rk1, pk1;
        nd.RP(k, rk, pk);
        nd.RP(k + 1, rk1, pk1);
        set_a_b_nodes(rj, mj, P, rk, pk, rk1, pk1, a, b);
    }
}
__device__ __forceinline__ void set_a_b(const double *__restrict__ r, const double *__restrict__ phi,
                                        double rj, double mj, const KParams &P, int64_t k,
                                        double *a, double *b)
{
    set_a_b_n(SplitNodes{r, phi}, rj, mj, P, k, a, b);
}

// cmc_nr.c:239-269 + :393-403: v_r^2 inside [r_k, r_{k+1}]; cen = cenma.m * madhoc
__device__ __forceinline__ double vr2_in_interval(const double *__restrict__ r, const double *__restrict__ phi,
                                                  double rj, double mj, double inv_nstar, double cen, int64_t k,
                                                  double E, double J, double x)
{
    const double eps = 2.220446049250313e-16;
    double pot;
    if (fabs(x - r[k]) < eps) pot = phi[k];
    else if (fabs(x - r[k + 1]) < eps) pot = phi[k + 1];
    else if (x < r[1]) pot = phi[0] - cen / x;
    else pot = (phi[k] + (phi[k + 1] - phi[k]) * (1.0 / r[k] - 1.0 / x) / (1.0 / r[k] - 1.0 / r[k + 1]));
    return function_q(rj, mj, inv_nstar, x, pot, E, J);
}

__device__ __forceinline__ bool interval_converged(double lo, double hi, double epsabs, double epsrel)
{
    double alo = fabs(lo), ahi = fabs(hi), min_abs;
    if ((lo > 0.0 && hi > 0.0) || (lo < 0.0 && hi < 0.0)) min_abs = alo < ahi ? alo : ahi;
    else min_abs = 0.0;
    return fabs(hi - lo) < epsabs + epsrel * min_abs;
}

// cmc_nr.c:500-603 find_root_vr by the Brent-Dekker method (Brent 1973, ch. 4),
// the same iteration as the CPU oracle's.  Rare fallback path; scalar arguments and a
// returned pair keep its caller's objects out of private memory.  (Not a call: around one
// the sampler spilled 30 registers, 128 B a star.)
struct RootVr { double root; int bad; };
__device__ __forceinline__ RootVr find_root_vr(const double *__restrict__ r, const double *__restrict__ phi,
                                            double rj, double mj, double inv_nstar, double cen, int64_t k,
                                            double E, double J)
{
    bool bad_ = false, *bad = &bad_;
    const double prec = 1e-11, deps = 2.220446049250313e-16;
    int iter = 100;
    double a = r[k], b = r[k + 1];
    double fa = vr2_in_interval(r, phi, rj, mj, inv_nstar, cen, k, E, J, a);
    double fb = vr2_in_interval(r, phi, rj, mj, inv_nstar, cen, k, E, J, b);
    if ((fa > 0) == (fb > 0) && (fa < 0) == (fb < 0)) return RootVr{0.0, 1};
    double c = a, fc = fa, d = b - a, e = d;
    double lo = a < b ? a : b, hi = a < b ? b : a;
    bool converged = false;
    double prev_apsis = -1.0;
    while (!converged && iter-- > 0) {
        if ((fb > 0 && fc > 0) || (fb < 0 && fc < 0)) { c = a; fc = fa; d = b - a; e = d; }
        if (fabs(fc) < fabs(fb)) { a = b; b = c; c = a; fa = fb; fb = fc; fc = fa; }
        double tol = 2.0 * deps * fabs(b);
        double mm = 0.5 * (c - b);
        if (fb == 0.0) { lo = hi = b; converged = true; break; }
        if (fabs(e) < tol || fabs(fa) <= fabs(fb)) {
            d = mm; e = mm;
        } else {
            double p, q, r2, s2 = fb / fa;
            if (a == c) {
                p = 2.0 * mm * s2; q = 1.0 - s2;
            } else {
                q = fa / fc; r2 = fb / fc;
                p = s2 * (2.0 * mm * q * (q - r2) - (b - a) * (r2 - 1.0));
                q = (q - 1.0) * (r2 - 1.0) * (s2 - 1.0);
            }
            if (p > 0) q = -q; else p = -p;
            if (2.0 * p < fmin(3.0 * mm * q - fabs(tol * q), fabs(e * q))) { e = d; d = p / q; }
            else { d = mm; e = mm; }
        }
        a = b; fa = fb;
        if (fabs(d) > tol) b += d;
        else b += (mm > 0 ? tol : -tol);
        fb = vr2_in_interval(r, phi, rj, mj, inv_nstar, cen, k, E, J, b);
        lo = b < c ? b : c; hi = b < c ? c : b;
        if ((fb > 0 && fc > 0) || (fb < 0 && fc < 0)) { lo = a < b ? a : b; hi = a < b ? b : a; }
        converged = interval_converged(lo, hi, prec, prec);
        if (!converged && iter < 10) {
            if (prev_apsis >= 0.0 && fabs(b - prev_apsis) < 5e-13 + 5e-13 * fabs(b)) converged = true;
            prev_apsis = b;
        }
    }
    if (!converged) *bad = true;
    double apsis = b;
    if (vr2_in_interval(r, phi, rj, mj, inv_nstar, cen, k, E, J, apsis) < 0.) {
        if (vr2_in_interval(r, phi, rj, mj, inv_nstar, cen, k, E, J, lo) < 0.) apsis = hi;
        if (vr2_in_interval(r, phi, rj, mj, inv_nstar, cen, k, E, J, hi) < 0.) apsis = lo;
    }
    if (vr2_in_interval(r, phi, rj, mj, inv_nstar, cen, k, E, J, apsis) < 0.) *bad = true;
    return RootVr{apsis, bad_ ? 1 : 0};
}

// Top levels of the sorted-potential search tree staged in LDS: cr[s] = r[k(s)],
// cphi[s] = phi[k(s)] with k(s) = min(s * stride, n + 1), s = 0..cs (k(cs) = n + 1).
// Radial index of the sorted radii: bucket b of a radius x > 0 is
// (bits(x) - bits(r_1)) >> shift (the IEEE bits of a positive double order like the
// values), clamped to nb; t[b] = number of nodes k in 1..n whose bucket is below b
// (t has nb + 2 entries).  Every node up to t[b] lies below x and every node after
// t[b + 1] above it, so [t[b], t[b + 1] + 1] brackets the largest k with r_k < x.
struct RIdx {
    const uint32_t *t;
    uint64_t lo;
    int shift;
    uint32_t nb;
};
__device__ __forceinline__ int ridx_shift(uint64_t lo, uint64_t hi, int bits)
{
    const uint64_t d = hi > lo ? hi - lo : 0;
    const int len = d ? 64 - __clzll((long long)d) : 0;
    return len > bits ? len - bits : 0;
}
__device__ __forceinline__ uint32_t ridx_bucket(const RIdx &x, double r)
{
    const uint64_t u = (uint64_t)__double_as_longlong(r);
    const uint64_t d = u > x.lo ? (u - x.lo) >> x.shift : 0;
    return d < x.nb ? (uint32_t)d : x.nb;
}
// the index of nodes 1..n (packed (r, phi), n >= 1) with 2^bits buckets
__device__ __forceinline__ RIdx ridx_of(const uint32_t *t, const double2 *__restrict__ nodes, int64_t n, int bits)
{
    RIdx x;
    x.t = t;
    x.nb = 1u << bits;
    x.lo = (uint64_t)__double_as_longlong(nodes[1].x);
    x.shift = ridx_shift(x.lo, (uint64_t)__double_as_longlong(nodes[n].x), bits);
    return x;
}

// [lo, hi] with r_lo < x <= r_hi (x >= r_1, x <= r_{n+1})
__device__ __forceinline__ void ridx_bracket(const RIdx &x, double r, int32_t &lo, int32_t &hi)
{
    const uint32_t b = ridx_bucket(x, r);
    lo = (int32_t)x.t[b];
    hi = (int32_t)x.t[b + 1] + 1;
}

struct Coarse {
    const double *cr, *cphi;
    int64_t stride, n1;          // stride is a multiple of MID_STEP
    uint32_t inv_stride;         // 2^32 / stride, for coarse_s
    int cs;
    // middle level in global memory (L2-resident): (r, phi) at every MID_STEP-th node
    const double2 *mid;
    // learned bracket proposal: predicted log r_peri, log r_apo and the half-width
    bool hint;
    float lrp, lra, margin;
    // radial index (t == nullptr: not built)
    RIdx ri;
};

constexpr int MID_STEP = 16;

__device__ __forceinline__ int64_t coarse_stride(int64_t n, int cs)
{
    int64_t st = (n + 1 + cs - 1) / cs;
    st = (st + MID_STEP - 1) / MID_STEP * MID_STEP;
    return st < MID_STEP ? MID_STEP : st;
}

__device__ __forceinline__ int64_t coarse_k(const Coarse &c, int s)
{
    int64_t k = (int64_t)s * c.stride;
    return k < c.n1 ? k : c.n1;
}
__device__ __forceinline__ int32_t coarse_k32(const Coarse &c, int s)
{
    const int32_t k = s * (int32_t)c.stride;       // at most n + 1 + the stride
    return k < (int32_t)c.n1 ? k : (int32_t)c.n1;
}
// k / stride: the truncated reciprocal gives the quotient or one less
__device__ __forceinline__ int coarse_s(const Coarse &c, int32_t k)
{
    const uint32_t q = __umulhi((uint32_t)k, c.inv_stride), st = (uint32_t)c.stride;
    return (int)(q + ((uint32_t)k - q * st >= st ? 1u : 0u));
}

// Largest t in [t0, t1] with eval(mid[t]) true, or t0 - 1 if there is none, for a
// predicate that is true then false over [t0, t1].  eval also returns a key, negative
// where the predicate holds, that varies smoothly with t; k_lo and k_hi are the keys
// just outside the range (at the bracket ends, k_lo < 0 <= k_hi).  Up to two probes
// read a whole 128-byte line of the middle table (8 entries) at the index where the
// keys interpolate to zero; the rest is bisection.  The answer is the same for any
// guesses, since the predicate alone decides it.
template <class Eval>
__device__ __forceinline__ int64_t mid_search(const double2 *__restrict__ mid, int64_t t0, int64_t t1, double k_lo,
                                              double k_hi, Eval eval)
{
    int64_t lo = t0 - 1, hi = t1 + 1;         // eval true at lo, false at hi (virtually)
    for (int probe = 0; probe < 2 && hi - lo > 1; probe++) {
        double f = k_lo / (k_lo - k_hi);
        if (!(f > 0.0 && f < 1.0)) f = 0.5;   // also NaN
        int64_t g = lo + 1 + (int64_t)(f * (double)(hi - lo - 1));
        if (g >= hi) g = hi - 1;
        const int64_t ls = g & ~(int64_t)7;
        int64_t last_true = lo, first_false = hi;
        double kt = k_lo, kf = k_hi;
        double2 e[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int64_t t = ls + u;
            if (t > lo && t < hi) e[u] = mid[t];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int64_t t = ls + u;
            if (t > lo && t < hi && first_false == hi) {
                double k;
                if (eval(e[u], k)) { last_true = t; kt = k; }
                else { first_false = t; kf = k; }
            }
        }
        lo = last_true; k_lo = kt;
        hi = first_false; k_hi = kf;
    }
    while (hi - lo > 1) {
        const int64_t m = lo + ((hi - lo) >> 1);
        double k;
        if (eval(mid[m], k)) lo = m;
        else hi = m;
    }
    return lo;
}

// potential(x) with the index search started from the LDS samples: the result is the
// unique largest k with r[k] < x, so any bracket [lo, hi] with r[lo] < x <= r[hi]
// gives the same index as the full-range search.
template <class N>
__device__ __forceinline__ double potential_at_coarse_n(const N &nd, int64_t n_max, double x, int64_t lo, int64_t hi,
                                                        const Coarse &c, bool *bad, int32_t *k_out = nullptr)
{
    if (x == 0.0 || x < nd.R(1)) return potential_at_n(nd, n_max, x, lo, hi, bad, k_out);
    int a = 0, b = c.cs;                    // largest s with cr[s] < x (cr[0] = r[0] < x)
    while (a < b) {
        int m = (a + b + 1) >> 1;
        if (c.cr[m] < x) a = m;
        else b = m - 1;
    }
    const float lx = __logf((float)x);
    double k_lo = -1.0, k_hi = 1.0;
    if (a < c.cs) {
        int64_t ka = coarse_k(c, a), kb = coarse_k(c, a + 1);
        if (ka > lo) lo = ka;
        if (kb < hi) hi = kb;
        k_lo = (double)(__logf((float)c.cr[a]) - lx);
        k_hi = (double)(__logf((float)c.cr[a + 1]) - lx);
    }
    if (c.mid) {
        // largest mid node strictly inside (lo, hi) with r < x
        const int64_t t0 = (lo + MID_STEP) / MID_STEP, t1 = (hi - 1) / MID_STEP;
        if (t0 <= t1) {
            const int64_t t = mid_search(c.mid, t0, t1, k_lo, k_hi, [&](double2 e, double &k) {
                k = (double)(__logf((float)e.x) - lx);
                return e.x < x;
            });
            if (t < t0) {
                hi = MID_STEP * t0;
            } else {
                lo = MID_STEP * t;
                if (MID_STEP * (t + 1) < hi) hi = MID_STEP * (t + 1);
            }
        }
    }
    return potential_at_n(nd, n_max, x, lo, hi, bad, k_out);
}
// potential(x) through the radial index: the node below x's bucket and the two after it
// (one index word, then three node loads that do not wait for each other) hold the
// interval unless the bucket holds more nodes, which a bisection up to the next bucket's
// first node settles.  The interval is the unique largest i with r_i < x that the
// full-range search returns.  r1: the innermost radius.
__device__ __forceinline__ double potential_at_ridx(const double2 *__restrict__ nodes, int64_t n_max, double r1, double x,
                                                    const RIdx &ri, bool *bad, int32_t *k_out)
{
    const PackedNodes nd{nodes};
    if (x == 0.0 || x < r1) return potential_at_n(nd, n_max, x, 1, n_max + 1, bad, k_out);
    const uint32_t b = ridx_bucket(ri, x);
    int32_t i = (int32_t)ri.t[b];
    const double2 *__restrict__ at = nodes + i;              // nodes holds two entries past n_max + 1
    double2 u = at[0], v = at[1];
    const double2 w = at[2];
    if (!(i >= n_max || v.x >= x)) {
        if (w.x >= x) {
            i++;
            u = v;
            v = w;
        } else {
            const int32_t hi = (int32_t)ri.t[b + 1] + 1;
            i = i + 2 >= hi - 1 ? i + 2 : (int32_t)find_zero_r_n(nd, i + 2, hi, x);
            u = nodes[i];
            v = nodes[i + 1];
        }
    }
    *k_out = i;
    if (u.x > x || v.x < x) { *bad = true; return 0.0; }
    if (i == 0) return v.y;
    return u.y + (v.y - u.y) * (1.0 / u.x - 1.0 / x) / (1.0 / u.x - 1.0 / v.x);
}

// A guess of the radius where Q changes sign between nodes (ra, pa) and (rb, pb),
// ra < rb: the potential between them taken as the Henon interpolant A/r + B through
// the two nodes (exactly the reference's interpolation when they are adjacent) plus
// the star's own term (m_j/r_j below r_j, m_j/r above; judged at ra), so that
// Q r^2 = 2(E - B - s0) r^2 - 2(A + s1) r - J^2.  The smaller positive root for the
// pericentre, the larger for the apocentre; negative or NaN when there is none.  Only a
// guess: every index it leads to is verified by the signs of Q.  So its reciprocals and root
// are the hardware's estimates and one Newton step: where that is not enough, the guess is a
// node or two off, or outside the bracket, and costs a probe.
__device__ __forceinline__ double rcp_guess(double x)
{
    const double y = __builtin_amdgcn_rcp(x);
    return __builtin_fma(y, __builtin_fma(-x, y, 1.0), y);
}
__device__ __forceinline__ double interp_root(const QStar &q, double ra, double pa, double rb, double pb, bool peri)
{
    const double A = (pb - pa) * ra * (rb * rcp_guess(ra - rb)), B = pa - A * rcp_guess(ra);
    const bool out = ra >= q.rj;
    const double h2 = q.E - B - (out ? 0.0 : q.s0), h1 = A + (out ? q.s1 : 0.0);
    const double disc = __builtin_fma(h1, h1, 2.0 * h2 * q.J2);         // roots of 2 h2 r^2 - 2 h1 r - J^2
    const double y = __builtin_amdgcn_rsq(disc);
    double sq = disc * y;
    sq = __builtin_fma(__builtin_fma(-sq, sq, disc), 0.5 * y, sq);
    const double w = h1 + (h1 >= 0.0 ? sq : -sq);
    const double x1 = 0.5 * w * rcp_guess(h2), x2 = -q.J2 * rcp_guess(w);
    const double lo = x1 < x2 ? x1 : x2, hi = x1 < x2 ? x2 : x1;
    return peri && lo > 0.0 ? lo : hi;
}

// find_zero_Q's answer on a bracket [lo, hi] whose ends have the bisection's
// predicate true and false (POSITIVE: the apocentre, predicate Q > 0; otherwise the
// pericentre, Q < 0), for a Q with one sign change on the bracket: interpolation
// steps (interp_root on the current bracket ends, turned into a node by the radial index,
// that node and the two after it loaded together and probed in order) narrow it, then a
// bisection in the nodes finishes.  Every index kept is a probed node, so the answer is
// the unique sign change, the index the full-range bisection returns.  (rl, pl), (rh, ph):
// nodes lo and hi on entry, nodes k and k + 1 of the answer k on return: the caller reads
// no node again.  (The sampler is bound by the rate of such gathers, 64 lines to a wave's
// load; probing the two ends of the index's bracket, with its ends and the answer's nodes
// read for themselves, took about 12 a search, this about 5.)
template <bool POSITIVE>
__device__ __forceinline__ int32_t ridx_zero_Q(const double2 *__restrict__ nodes, const RIdx &ri, const QStar &q,
                                               int32_t lo, int32_t hi, double &rl, double &pl, double &rh, double &ph)
{
    int32_t l = lo, h = hi;
    // node k probed: true when the bracket's lower end moved to it
    auto probe = [&](int32_t k, const double2 &v) {
        const int sg = q_sign(q, v.x, v.y);
        const bool in = POSITIVE ? q_gt0(sg) : q_lt0(sg);
        if (in) { l = k; rl = v.x; pl = v.y; }
        else { h = k; rh = v.x; ph = v.y; }
        return in;
    };
    for (int it = 0; it < 3 && h - l > 1; it++) {
        const double rg = interp_root(q, rl, pl, rh, ph, !POSITIVE);
        int32_t a = l + ((h - l) >> 1);            // no usable guess: a bisection step
        if (rg > rl && rg < rh) {
            const int32_t g = (int32_t)ri.t[ridx_bucket(ri, rg)];
            a = g < l ? l : (g > h - 1 ? h - 1 : g);
        }
        const double2 u = nodes[a], v = nodes[a + 1], w = nodes[a + 2];
        if ((a == l || probe(a, u)) && a + 1 < h && probe(a + 1, v) && a + 2 < h) probe(a + 2, w);
    }
    while (h - l > 1) {
        const int32_t m = l + ((h - l) >> 1);
        probe(m, nodes[m]);
    }
    return l;
}

struct OrbitRS { double rp, ra, dQdrp, dQdra; int64_t kmin, kmax; int circular; int brent; int linscan; int err;
                 int hint_hits, hint_misses; };

// cmc_orbit.c:413-540 calc_orbit_new after get_positive_Q_index has produced ktemp
// (an index with Q > 0; ktemp < 0 means "no positive Q": circular orbit).
// HAS_C: the LDS samples, radial index and learned proposal of Cr are available, and pj is
// phi at j, q the star's QStar.  (A template flag rather than a null test of a pointer: comparing the address
// of a private object with null is not folded on this target and keeps the object in
// scratch memory.)
template <class N, bool HAS_C>
__device__ __forceinline__ OrbitRS calc_orbit_core(const N &nd, const double *__restrict__ r,
                                                   const double *__restrict__ phi, int64_t n_max, int64_t j,
                                                   double rj, double mj, const KParams &P, double E, double J,
                                                   int64_t ktemp, const Coarse &Cr, const QStar &q, double pj = 0.0)
{
    OrbitRS o;
    o.brent = 0; o.linscan = 0; o.err = 0; o.hint_hits = 0; o.hint_misses = 0;
    if (ktemp < 0) {
        o.rp = o.ra = rj; o.kmin = o.kmax = j; o.dQdrp = o.dQdra = 0.0; o.circular = 1;
        return o;
    }
    int64_t kmin, kmax;
    double rp0, pp0, rp1, pp1;         // nodes kmin, kmin + 1
    double ra0, pa0, ra1, pa1;         // nodes kmax, kmax + 1
    if constexpr (HAS_C) {
        // Q is negative at the centre, positive on one interval around ktemp (= j here) and
        // negative far out (r^3 dPhi/dr = r M(r) increases), so the index bisection's result
        // is the unique sign change of its bracket; the LDS samples narrow both brackets
        // to one sample interval before the interpolation search in global memory.
        const int32_t kt = (int32_t)ktemp, n1 = (int32_t)n_max + 1;
        int32_t kp_lo = 0, kp_hi = kt, ka_lo = kt, ka_hi = n1;
        bool got_p = false, got_a = false;
        bool vp = false, va = false;   // bracket ends checked: Q(lo), Q(hi) have the bisection's signs
        rp1 = ra0 = rj;
        pp1 = pa0 = pj;
        if (Cr.hint) {
            // learned proposals: the index range of the predicted apsis +- margin (in
            // log r), accepted only when Q has the bisection's signs at its ends
            const float ep = __expf(Cr.margin);
            int32_t a, b;
            ridx_bracket(Cr.ri, (double)(__expf(Cr.lrp) / ep), a, b);
            int32_t lo = a < 0 ? 0 : a;
            ridx_bracket(Cr.ri, (double)(__expf(Cr.lrp) * ep), a, b);
            int32_t hi = b > kt ? kt : b;
            if (lo < hi && q_lt0(q_sign(q, nd.R(lo), nd.P(lo))) &&
                (hi == kt || q_ge0(q_sign(q, nd.R(hi), nd.P(hi))))) {
                kp_lo = lo; kp_hi = hi; got_p = vp = true; o.hint_hits++;
            } else {
                o.hint_misses++;
            }
            ridx_bracket(Cr.ri, (double)(__expf(Cr.lra) / ep), a, b);
            lo = a < kt ? kt : a;
            ridx_bracket(Cr.ri, (double)(__expf(Cr.lra) * ep), a, b);
            hi = b > n1 ? n1 : b;
            if (lo < hi && (lo == kt || q_gt0(q_sign(q, nd.R(lo), nd.P(lo)))) &&
                !q_gt0(q_sign(q, nd.R(hi), nd.P(hi)))) {
                ka_lo = lo; ka_hi = hi; got_a = va = true; o.hint_hits++;
            } else {
                o.hint_misses++;
            }
            // a verified learned bracket is narrowed by the LDS samples inside it: the
            // sample bisection runs over those samples only
            auto narrow = [&](int32_t &lo, int32_t &hi, bool positive) {
                const int s0 = coarse_s(Cr, lo) + 1, s1 = coarse_s(Cr, hi - 1);
                if (s0 > s1 || s1 > Cr.cs) return;
                int a = s0 - 1, b = s1;                    // sample a: predicate true (a = s0 - 1: node lo)
                while (a < b) {
                    const int m = (a + b + 1) >> 1;
                    const int sg = q_sign(q, Cr.cr[m], Cr.cphi[m]);
                    if (positive ? q_gt0(sg) : q_lt0(sg)) a = m;
                    else b = m - 1;
                }
                if (a >= s0) lo = coarse_k32(Cr, a);
                if (a < s1) hi = coarse_k32(Cr, a + 1);
            };
            if (got_p) {
                narrow(kp_lo, kp_hi, false);
                nd.RP(kp_lo, rp0, pp0);
                nd.RP(kp_hi, rp1, pp1);
            }
            if (got_a) {
                narrow(ka_lo, ka_hi, true);
                nd.RP(ka_lo, ra0, pa0);
                nd.RP(ka_hi, ra1, pa1);
            }
        }
        if (!got_p && kt >= 1 && q_lt0(q_sign(q, Cr.cr[0], Cr.cphi[0]))) {
            int a = 0, b = coarse_s(Cr, kt - 1);
            const int top = b;
            while (a < b) {
                int m = (a + b + 1) >> 1;
                if (q_lt0(q_sign(q, Cr.cr[m], Cr.cphi[m]))) a = m;
                else b = m - 1;
            }
            kp_lo = coarse_k32(Cr, a);
            rp0 = Cr.cr[a];
            pp0 = Cr.cphi[a];
            if (a < top) {
                kp_hi = coarse_k32(Cr, a + 1);
                rp1 = Cr.cr[a + 1];
                pp1 = Cr.cphi[a + 1];
            }
            vp = true;
        }
        const int sb = coarse_s(Cr, kt) + 1;
        if (!got_a && sb <= Cr.cs && !q_gt0(q_sign(q, Cr.cr[Cr.cs], Cr.cphi[Cr.cs]))) {
            va = true;
            int a = sb - 1, b = Cr.cs - 1;                 // sample a: Q > 0 (a = sb - 1: node ktemp)
            while (a < b) {
                int m = (a + b + 1) >> 1;
                if (q_gt0(q_sign(q, Cr.cr[m], Cr.cphi[m]))) a = m;
                else b = m - 1;
            }
            if (a >= sb) {
                ka_lo = coarse_k32(Cr, a);
                ra0 = Cr.cr[a];
                pa0 = Cr.cphi[a];
            }
            ka_hi = coarse_k32(Cr, a + 1);
            ra1 = Cr.cr[a + 1];
            pa1 = Cr.cphi[a + 1];
        }
        // verified brackets: interpolation search through the radial index; otherwise the
        // full-range bisection (which also settles the direction itself)
        const double2 *nodes = nd.rp;
        if (vp) {
            kmin = ridx_zero_Q<false>(nodes, Cr.ri, q, kp_lo, kp_hi, rp0, pp0, rp1, pp1);
        } else {
            kmin = find_zero_Q_n(nd, rj, mj, P.inv_nstar, kp_lo, kp_hi, E, J);
            if (kmin >= 0) {
                nd.RP(kmin, rp0, pp0);
                nd.RP(kmin + 1, rp1, pp1);
            }
        }
        if (va) {
            kmax = ridx_zero_Q<true>(nodes, Cr.ri, q, ka_lo, ka_hi, ra0, pa0, ra1, pa1);
        } else {
            kmax = find_zero_Q_n(nd, rj, mj, P.inv_nstar, ka_lo, ka_hi, E, J);
            if (kmax >= 0) {
                nd.RP(kmax, ra0, pa0);
                nd.RP(kmax + 1, ra1, pa1);
            }
        }
    } else {
        kmin = find_zero_Q_n(nd, rj, mj, P.inv_nstar, 0, ktemp, E, J);
        kmax = find_zero_Q_n(nd, rj, mj, P.inv_nstar, ktemp, n_max + 1, E, J);
        if (kmin >= 0 && kmax >= 0) {
            nd.RP(kmin, rp0, pp0);
            nd.RP(kmin + 1, rp1, pp1);
            nd.RP(kmax, ra0, pa0);
            nd.RP(kmax + 1, ra1, pa1);
        }
    }
    if (kmin < 0 || kmax < 0) {
        o.err = CMCG_E_BRACKET;
        o.rp = o.ra = rj; o.kmin = o.kmax = j; o.dQdrp = o.dQdra = 0.0; o.circular = 1;
        return o;
    }
    double ap, aa, b, rmin, rmax;
    if (kmin == 0) set_a_b_n(nd, rj, mj, P, 0, &ap, &b);
    else set_a_b_nodes(rj, mj, P, rp0, pp0, rp1, pp1, &ap, &b);
    double inside_sqrt = ap * ap - 2.0 * J * J * (b - E);
    if (inside_sqrt < 0.0) rmin = -1.0 * J * J / ap;
    else rmin = J * J / (-ap + sqrt(inside_sqrt));
    const bool brent_p = inside_sqrt < 0.0 && ((rmin < rp0) || (rmin > rp1));
    if (kmax == 0) set_a_b_n(nd, rj, mj, P, 0, &aa, &b);
    else set_a_b_nodes(rj, mj, P, ra0, pa0, ra1, pa1, &aa, &b);
    inside_sqrt = aa * aa - 2.0 * J * J * (b - E);
    if (inside_sqrt < 0.0) rmax = -aa / (2.0 * (b - E));
    else rmax = (-aa + sqrt(inside_sqrt)) / (2.0 * (b - E));
    const bool brent_a = inside_sqrt < 0.0 && ((rmax < ra0) || (rmax > ra1));
    if (brent_p || brent_a) {
        o.brent = 1;
#pragma unroll 1
        for (int side = 0; side < 2; side++) {
            if (!(side ? brent_a : brent_p)) continue;
            const RootVr rv = find_root_vr(r, phi, rj, mj, P.inv_nstar, P.cenma_m * P.madhoc, side ? kmax : kmin, E, J);
            if (rv.bad) o.err = CMCG_E_BRENT;
            if (side) rmax = rv.root;
            else rmin = rv.root;
        }
    }
    const double dQdr_min = 2.0 * J * J / (rmin * rmin * rmin) + 2.0 * ap / (rmin * rmin);
    const double dQdr_max = 2.0 * J * J / (rmax * rmax * rmax) + 2.0 * aa / (rmax * rmax);
    if ((rmin > rmax) || (dQdr_min <= 0.) || (dQdr_max >= 0.)) {
        o.rp = o.ra = rj; o.kmin = o.kmax = j; o.dQdrp = o.dQdra = 0.0; o.circular = 1;
    } else {
        o.rp = rmin; o.ra = rmax; o.kmin = kmin; o.kmax = kmax;
        o.dQdrp = dQdr_min; o.dQdra = dQdr_max; o.circular = 0;
    }
    return o;
}

template <class N>
__device__ __forceinline__ OrbitRS calc_orbit_from_n(const N &nd, const double *__restrict__ r,
                                                     const double *__restrict__ phi, int64_t n_max, int64_t j,
                                                     double rj, double mj, const KParams &P, double E, double J,
                                                     int64_t ktemp)
{
    const Coarse none{};
    const QStar unused{};
    return calc_orbit_core<N, false>(nd, r, phi, n_max, j, rj, mj, P, E, J, ktemp, none, unused);
}

__device__ __forceinline__ OrbitRS calc_orbit_from(const double *__restrict__ r, const double *__restrict__ phi,
                                                   int64_t n_max, int64_t j, double rj, double mj,
                                                   const KParams &P, double E, double J, int64_t ktemp)
{
    return calc_orbit_from_n(SplitNodes{r, phi}, r, phi, n_max, j, rj, mj, P, E, J, ktemp);
}

// get_positive_Q_index (cmc_orbit.c:30-59) with its linear scan, then calc_orbit_from.
// Used by the small batch entry points; the orbit phase defers the scan instead.
__device__ __forceinline__ OrbitRS calc_orbit(const double *__restrict__ r, const double *__restrict__ phi,
                                              int64_t n_max, int64_t j, double rj, double mj,
                                              const KParams &P, double E, double J)
{
    int64_t ktemp = j;
    double Qtemp = function_q(rj, mj, P.inv_nstar, r[ktemp], phi[ktemp], E, J);
    int lin = 0;
    if (Qtemp <= 0.0) {
        lin = 1;
        ktemp = -1;
        do {
            ktemp++;
            Qtemp = function_q(rj, mj, P.inv_nstar, r[ktemp], phi[ktemp], E, J);
        } while (Qtemp <= 0.0 && ktemp <= n_max);
        if (ktemp >= n_max) ktemp = -1;            // cmc_orbit.c:52-56
    }
    OrbitRS o = calc_orbit_from(r, phi, n_max, j, rj, mj, P, E, J, ktemp);
    o.linscan = lin;
    return o;
}

// ---------------------------------------------------------------- host side
struct cmcg_ctx_impl;   // defined in cmcg_api.hip

#define CMCG_HIP_CHECK(expr)                                                       \
    do {                                                                           \
        hipError_t _e = (expr);                                                    \
        if (_e != hipSuccess) { cmcg_report_hip(_e, #expr, __FILE__, __LINE__); return CMCG_E_HIP; } \
    } while (0)

void cmcg_report_hip(hipError_t e, const char *expr, const char *file, int line);
