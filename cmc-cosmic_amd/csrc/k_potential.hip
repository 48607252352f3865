// a2: potential_calculate (src/cmc/cmc_utils.c:675-736), reproducing the reference's
// sequential FP64 rounding bit for bit with parallel scans.
//
// The reference evaluates three floating-point chains one element at a time:
//   A  mprev += m_k                  k = 1..N          (total mass, :685-696)
//   B  mprev -= m_k / N_STAR         k = N..2          (enclosed mass M_k, :723)
//   C  phi_k = phi_{k+1} - M_k (1/r_k - 1/r_{k+1})     (:722)
// Each chain is v_j = fl(v_{j-1} + s*x_j) and is monotone.  Repeated rounding makes
// the result drift from the exact sums (6e-11 relative at N = 1e5), so a correctly
// rounded parallel scan does not reproduce it.  Exact reproduction uses:
//
// * If v_{j-1} and v_j lie in one binade with ulp u, then fl(v_{j-1} + s x_j) =
//   v_{j-1} + RN_u(s x_j) unless s x_j / u is a tie: the increment does not depend
//   on v_{j-1}.  Such "regular" elements are recognised from a double estimate of
//   the prefix sums of the x and a rigorous bound on its error and on the chain's
//   own accumulated rounding; the rest ("sensitive": binade crossings, ties, tiny
//   values) are few, about one per binade.
// * Segment and walk: a regular increment is an integer R in units of its binade's
//   ulp, and a run of them between two sensitive elements stays in one binade, so
//   an int64 scan that restarts at every sensitive element gives each run's exact
//   sum.  One thread or wave walks the sensitive elements in order, each getting
//   fl(v_prev + s x) from the exact value before it (the previous one plus the run
//   in between), then every element is rebuilt in parallel from the last sensitive
//   value before it.  Four passes: tile sums (fused into the kernel that produces
//   the increments), classification, walk, rebuild.
// * Every element of chains B and C, and of the reports' chains, is rebuilt and verified
//   against fl(v_{j-1} + s x_j), so there the estimate's bound decides only the speed, never
//   the result.  A violation (only when the bound is exceeded, or a report's list; the
//   potential's hold every star) is repaired by running the recurrence itself.
// * Chain A needs only its last value and is not rebuilt: its exactness rests on the bound
//   (err_bound), which is rigorous for masses that are not negative and finite (any other mass
//   sends all three chains to the repair).
#include "kernels.hpp"

namespace {
constexpr int CT = 256;             // threads per tile
constexpr int CI = 8;               // items per thread
constexpr int CTILE = CT * CI;
constexpr int RAW_CAP = 2048;         // sensitive elements that the walk puts in order in LDS (more: in memory)
constexpr int WALK_T = 1024;          // threads of the one-block kernels
constexpr int WALK_CHUNK = 256;       // sensitive elements staged per round of the walk
constexpr int WALK_REG = 16;          // tiles per walk thread held in registers (N <= 8.4e6 at CT*CI = 2048)

// ---------------------------------------------------------------- segment and walk
// The classification needs only the binade of each chain value, so it runs on a
// double estimate of the prefix sums with a rigorous error bound.  A regular element
// adds RN_u(s x) = R u, u = 2^(b-52) the ulp of its binade b, and all regular
// elements between two sensitive ones share one binade: a sum of the integers R that
// restarts at every sensitive element (a segmented scan) is exact in int64, and times
// u exact in double.
struct EsaArgs {
    const double *x;
    double *g;
    double sign;
    const double *v0p;
    int64_t *first_bad;         // [1] first element that violates the recurrence (L: none)
    const int64_t *Lp;
    int slack;                  // error bound widened by 2^slack (0; a test hook raises it)
    int64_t extra;              // the start value is only an estimate, as uncertain as this many more elements
    // per tile
    double *tsumP, *tpreP;      // estimated sums of s*x and their exclusive prefixes
    int64_t *tcnt, *ttail;      // sensitive count; regular sum after the tile's last sensitive element
    int64_t *toff, *tcarry;     // sensitive elements before the tile; regular sum of the segment open at its start
    // the sensitive elements in chain order
    int64_t *s_idx;
    double *s_pre;              // regular sum between the previous sensitive element and this one
    double *s_v;                // chain value after the element
    int64_t *s_n;               // count (uncapped)
    int64_t smax;               // capacity
    // appended by the classification in any order (raw_cap entries): index, regular sum
    // since the previous sensitive element of its tile (or the tile start), binade
    // before it (raw_bp), its number among the tile's (raw_bp + raw_cap) and its s x
    int64_t *raw_n, *raw_idx, *raw_part;
    int32_t *raw_bp;
    double *raw_sx;
    int64_t raw_cap;
};

// A run of elements: regular sum after its last sensitive element (all of it when it
// has none) and its number of sensitive elements.
struct Seg {
    int64_t sum;
    int64_t cnt;
};
// a followed by b
__device__ __forceinline__ Seg seg_then(Seg a, Seg b) { return Seg{b.cnt ? b.sum : a.sum + b.sum, a.cnt + b.cnt}; }
__device__ __forceinline__ Seg shfl_up_seg(Seg s, int d)
{
    return Seg{__shfl_up(s.sum, d, 64), __shfl_up(s.cnt, d, 64)};
}

// Block-wide exclusive scans (every thread of the block calls; lds holds blockDim/64
// entries).  The wave totals are folded in wave order, so the results do not depend
// on timing.
__device__ double block_excl_sum(double v, double *lds, double *total)
{
    const int t = threadIdx.x, lane = t & 63, w = t >> 6, nw = blockDim.x >> 6;
    double x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const double y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    double ex = __shfl_up(x, 1, 64);
    if (lane == 0) ex = 0.0;
    if (lane == 63) lds[w] = x;
    __syncthreads();
    double off = 0.0, tot = 0.0;
    for (int q = 0; q < nw; q++) {
        const double s = lds[q];
        if (q < w) off += s;
        tot += s;
    }
    *total = tot;
    __syncthreads();
    return off + ex;
}

// by a group of CT threads (a block, or half a block that gives each half its own lds)
__device__ Seg block_excl_seg(Seg v, Seg *lds, Seg *total)
{
    const int t = threadIdx.x % CT, lane = t & 63, w = t >> 6, nw = CT >> 6;
    Seg x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const Seg y = shfl_up_seg(x, d);
        if (lane >= d) x = seg_then(y, x);
    }
    Seg ex = shfl_up_seg(x, 1);
    if (lane == 0) ex = Seg{0, 0};
    if (lane == 63) lds[w] = x;
    __syncthreads();
    Seg off{0, 0}, tot{0, 0};
    for (int q = 0; q < nw; q++) {
        const Seg s = lds[q];
        if (q < w) off = seg_then(off, s);
        tot = seg_then(tot, s);
    }
    *total = tot;
    __syncthreads();
    return seg_then(off, ex);
}

__device__ __forceinline__ int binade_of(double v)
{
    // exponent of a normal double, or INT_MIN for zero, subnormal, inf, nan
    uint64_t b = (uint64_t)__double_as_longlong(v);
    int e = (int)((b >> 52) & 0x7ff);
    return (e == 0 || e == 0x7ff) ? INT32_MIN : e - 1023;
}

// binade of every value within e of the estimate v, or INT32_MIN if they differ
__device__ __forceinline__ int interval_binade(double v, double e)
{
    double lo = v - e, hi = v + e;
    if (!(lo > 0.0) && !(hi < 0.0)) return INT32_MIN;
    int b1 = binade_of(lo), b2 = binade_of(hi);
    return b1 == b2 ? b1 : INT32_MIN;
}

// Bound on |v - P| for the estimate P of the chain value v after j elements: the
// chain's own j roundings (at most 2^-53 |v| each, |v| <= vmax for a monotone chain)
// and the roundings of the estimate's sums in any order (at most (j + 2) 2^-53
// (|v0| + sum |s x|) <= (j + 2) 2^-52 vmax), with a factor 2 to spare.  A chain that is verified
// element by element would only take the repair if it failed; the total mass (the potential's
// chain A) is not, and relies on it.
__device__ __forceinline__ double err_bound(int64_t j, double vmax, int slack)
{
    return ldexp(((double)j + 2.0) * vmax, slack - 50) * 1.001;
}

// binade of the chain value before element j, or INT32_MIN when its error interval
// straddles binades; before element 0 the value is v0 (exactly, when extra is 0)
__device__ __forceinline__ int start_binade(int64_t j, double v0, double P, int slack, int64_t extra)
{
    if (j == 0 && extra == 0) return interval_binade(v0, 0.0);
    return interval_binade(P, err_bound(j + extra, fmax(fabs(v0), fabs(P)), slack));
}

// regular increment of an element in units of 2^(bp-52), or sensitive: bp, bq are the
// binades before and after it
__device__ __forceinline__ bool classify(double sx, int bp, int bq, int64_t *R)
{
    if (bp == INT32_MIN || bp != bq) return true;
    const double y = ldexp(sx, 52 - bp);      // exact unless it underflows, far below 1/2
    const double fy = floor(y);
    if (y - fy == 0.5 || !(fabs(y) <= 9007199254740992.0)) return true;
    *R = (int64_t)rint(y);
    return false;
}

// One tile's items, CI consecutive per thread.
struct TileItems {
    double sx[CI];      // s x_j (exact: s = +-1)
    double pa[CI];      // estimate of the chain value after the item
    int64_t R[CI];      // regular increment in units of 2^(bp - 52), 0 if sensitive
    int bp[CI];         // binade before the item
    uint32_t sens;      // bit u: item u sensitive
};

// A tile staged through LDS so that global memory is read and written in coalesced
// rows (element i of the tile by thread i mod CT) while each thread works on CI
// consecutive elements; one pad double per 8 keeps the per-thread reads free of bank
// conflicts.
constexpr int TILE_LDS = CTILE + CTILE / 8;
__device__ __forceinline__ int tile_slot(int i) { return i + (i >> 3); }

// src(j): element j's x.  The loads are issued on their own, as early as the caller can:
// after a launch each misses L2, and a chain of such misses is what a small cluster's
// passes wait for.
template <class Src>
__device__ __forceinline__ void fetch_tile(const Src &src, int64_t base, int64_t L, double (&v)[CI])
{
#pragma unroll
    for (int u = 0; u < CI; u++) {
        const int64_t j = base + u * CT + threadIdx.x;
        v[u] = j < L ? src(j) : 0.0;
    }
}

__device__ __forceinline__ void spread_tile(const double (&v)[CI], double sign, double *tbuf, double (&sx)[CI])
{
    const int t = threadIdx.x;
#pragma unroll
    for (int u = 0; u < CI; u++) tbuf[tile_slot(u * CT + t)] = sign * v[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < CI; u++) sx[u] = tbuf[tile_slot(t * CI + u)];
}

// the reverse; tbuf must be free (every thread past its last read of it)
__device__ __forceinline__ void store_tile(double *__restrict__ g, int64_t base, int64_t L, double *tbuf,
                                           const double (&v)[CI])
{
    const int t = threadIdx.x;
#pragma unroll
    for (int u = 0; u < CI; u++) tbuf[tile_slot(t * CI + u)] = v[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < CI; u++) {
        const int i = u * CT + t;
        const int64_t j = base + i;
        if (j < L) g[j] = tbuf[tile_slot(i)];
    }
}

// Classification of one tile (items past the end are regular with R = 0), from the
// fetched elements (v) and the estimated prefixes before the tile and before the next one.  Every kernel
// classifies through this function on the same inputs, so they agree element for
// element; the binade at a tile start is taken from the same expression in both tiles
// that meet there.  Nearly always a thread's whole range of
// values lies in one binade, checked once with the bound at its last element: then
// only the ties remain to be found.
__device__ __forceinline__ void tile_classify(const EsaArgs &a, const double (&v)[CI], int64_t tile, int64_t L, double v0,
                                              TileItems &it, double *lds, double *tbuf, double pre_t, double pre_t1)
{
    const int64_t j0 = tile * CTILE + (int64_t)threadIdx.x * CI;
    spread_tile(v, a.sign, tbuf, it.sx);
    double acc = 0.0;
#pragma unroll
    for (int u = 0; u < CI; u++) acc += it.sx[u];
    double tot;
    const double E = block_excl_sum(acc, lds, &tot);
    const double P0 = v0 + (pre_t + E);
    double P = P0, Pmin = P0, Pmax = P0;
#pragma unroll
    for (int u = 0; u < CI; u++) {
        P = P + it.sx[u];
        it.pa[u] = P;
        Pmin = fmin(Pmin, P);
        Pmax = fmax(Pmax, P);
    }
    it.sens = 0;
    const int64_t jl = j0 + CI < L ? j0 + CI : L;           // one past the thread's last element
    const bool edge = jl < L && jl % CTILE == 0;             // the next element opens the next tile
    const double Pn = edge ? v0 + (pre_t1 + 0.0) : 0.0;
    // fast path: every value before and after the thread's elements in one binade
    int bt = INT32_MIN;
    if (j0 < L) {
        const double vmax = fmax(fabs(v0), fmax(fabs(Pmin), fabs(Pmax)));
        const double err = err_bound(jl + a.extra, vmax, a.slack);
        const double lo = fmin(Pmin, j0 == 0 ? v0 : Pmin) - err, hi = fmax(Pmax, j0 == 0 ? v0 : Pmax) + err;
        if (lo > 0.0 || hi < 0.0) {
            const int b1 = binade_of(lo), b2 = binade_of(hi);
            if (b1 == b2) bt = b1;
        }
        if (j0 == 0 && bt != start_binade(0, v0, v0, a.slack, a.extra)) bt = INT32_MIN;
        if (edge && bt != start_binade(jl, v0, Pn, a.slack, a.extra)) bt = INT32_MIN;
    }
    if (bt != INT32_MIN) {
#pragma unroll
        for (int u = 0; u < CI; u++) {
            it.R[u] = 0;
            it.bp[u] = bt;
            if (j0 + u < L && classify(it.sx[u], bt, bt, &it.R[u])) {
                it.sens |= 1u << u;
                it.R[u] = 0;
            }
        }
        return;
    }
    P = P0;
    int bp = start_binade(j0, v0, P, a.slack, a.extra);
#pragma unroll
    for (int u = 0; u < CI; u++) {
        const int64_t j = j0 + u;
        const double Pq = it.pa[u];
        it.R[u] = 0;
        it.bp[u] = bp;
        if (j < L) {
            const double Pe = edge && j + 1 == jl ? Pn : Pq;
            const int bq = start_binade(j + 1, v0, Pe, a.slack, a.extra);
            if (classify(it.sx[u], bp, bq, &it.R[u])) {
                it.sens |= 1u << u;
                it.R[u] = 0;
            }
            bp = bq;
        }
        P = Pq;
    }
}

__device__ __forceinline__ Seg items_seg(const TileItems &it)
{
    Seg s{0, 0};
#pragma unroll
    for (int u = 0; u < CI; u++) {
        if ((it.sens >> u) & 1) {
            s.sum = 0;
            s.cnt++;
        } else {
            s.sum += it.R[u];
        }
    }
    return s;
}

__device__ __forceinline__ double seg_value(int64_t sum, int bp)
{
    return sum == 0 || bp == INT32_MIN ? 0.0 : ldexp((double)sum, bp - 52);
}

// Tile sums of s*x (acc: this thread's share); block 0 also resets the chain's flags.
__device__ void esa_tile_sums(const EsaArgs &a, int64_t L, double acc, double *lds, uint32_t tile)
{
    double tot;
    block_excl_sum(acc, lds, &tot);
    if (threadIdx.x == 0) {
        a.tsumP[tile] = tot;
        if (tile == 0) {
            a.first_bad[0] = 0;
            a.first_bad[1] = L;
            *a.raw_n = 0;
        }
    }
}

// one block: exclusive prefixes of the nt tile sums, in tile order
struct esa_tile_scan_kernel {
    static constexpr int LB = WALK_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, EsaArgs a, int64_t nt)
{
    __shared__ double lds[WALK_T / 64];
    const int64_t chunk = (nt + WALK_T - 1) / WALK_T;
    const int64_t b0 = (int64_t)threadIdx.x * chunk;
    double s = 0.0;
    for (int64_t b = b0; b < b0 + chunk && b < nt; b++) s += a.tsumP[b];
    double tot;
    double run = block_excl_sum(s, lds, &tot);
    for (int64_t b = b0; b < b0 + chunk && b < nt; b++) {
        a.tpreP[b] = run;
        run += a.tsumP[b];
    }
}
};

struct esa_sum_kernel {
    static constexpr int LB = CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, EsaArgs a)
{
    __shared__ double lds[CT / 64];
    const int64_t L = *a.Lp;
    const int64_t base = (int64_t)kg_.bid * CTILE;
    double v[CI];
#pragma unroll
    for (int u = 0; u < CI; u++) {
        const int64_t j = base + u * CT + threadIdx.x;
        v[u] = j < L ? a.x[j] : 0.0;
    }
    double acc = 0.0;
#pragma unroll
    for (int u = 0; u < CI; u++)
        if (base + u * CT + threadIdx.x < L) acc += a.sign * v[u];
    esa_tile_sums(a, L, acc, lds, kg_.bid);
}
};

// The estimated prefixes of tile t and t + 1 (the sums of tsumP before them), by one
// block: thread i sums the tiles i, i + CT, ... in order, and the threads' sums are
// reduced by a fixed tree.  Tile t + 1's own block forms the same sums term for term
// (its thread t mod CT ends with tile t), so both blocks get the same bits.
constexpr int64_t SELF_PREFIX_MAX = 16384;    // tiles; beyond, a one-block scan forms them
__device__ __forceinline__ double tree_sum(double v, double *lds)
{
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) lds[w] = v;
    __syncthreads();
    double r = lds[0];
    for (int q = 1; q < (int)(blockDim.x >> 6); q++) r += lds[q];
    __syncthreads();
    return r;
}
__device__ void tile_prefixes(const double *__restrict__ tsumP, int64_t t, double *lds, double *pre_t, double *pre_t1)
{
    double p = 0.0;
    for (int64_t q = threadIdx.x; q < t; q += CT) p += tsumP[q];
    const double p1 = (int64_t)threadIdx.x == t % CT ? p + tsumP[t] : p;
    *pre_t = tree_sum(p, lds);
    *pre_t1 = tree_sum(p1, lds);
}

// elements as they lie in memory
struct ArraySrc {
    const double *__restrict__ x;
    __device__ __forceinline__ double operator()(int64_t j) const { return x[j]; }
};

// LDS of the classification and the rebuild
struct ChainLds {
    double d[CT / 64];
    Seg s[CT / 64];
    double tbuf[TILE_LDS];
    double lastv[CT];
};

// One tile classified: its segment aggregate, and its sensitive elements appended to the
// chain's list.  v0: the start value (or its estimate).  Returns false in a thread that
// holds an element below zero, infinite or NaN.
__device__ __forceinline__ bool classify_tile(const EsaArgs &a, const double (&v)[CI], int64_t tile, int64_t L, double v0,
                                              double pre_t, double pre_t1, ChainLds &sh)
{
    TileItems it;
    tile_classify(a, v, tile, L, v0, it, sh.d, sh.tbuf, pre_t, pre_t1);
    bool ok = true;
#pragma unroll
    for (int u = 0; u < CI; u++) ok = ok && a.sign * it.sx[u] >= 0.0 && a.sign * it.sx[u] < __builtin_inf();
    Seg tot;
    const Seg pre = block_excl_seg(items_seg(it), sh.s, &tot);
    if (threadIdx.x == 0) {
        a.tcnt[tile] = tot.cnt;
        a.ttail[tile] = tot.sum;
    }
    if (!it.sens) return ok;
    int64_t cur = pre.sum, k = pre.cnt;
    const int64_t j0 = tile * CTILE + (int64_t)threadIdx.x * CI;
    int64_t slot = (int64_t)atomicAdd((unsigned long long *)a.raw_n, (unsigned long long)__popc(it.sens));
    for (int u = 0; u < CI; u++) {
        if ((it.sens >> u) & 1) {
            if (slot < a.raw_cap) {
                a.raw_idx[slot] = j0 + u;
                a.raw_part[slot] = cur;
                a.raw_bp[slot] = it.bp[u];
                a.raw_bp[a.raw_cap + slot] = (int32_t)k;
                a.raw_sx[slot] = it.sx[u];
            }
            slot++;
            k++;
            cur = 0;
        } else {
            cur += it.R[u];
        }
    }
    return ok;
}

// the estimated prefixes of a tile and the next: formed here (and this tile's stored in
// tpreP for the later passes), or read from tpreP (esa_tile_scan_kernel)
__device__ __forceinline__ void get_prefixes(const EsaArgs &a, int64_t tile, int self_prefix, double *lds, double *pre_t,
                                             double *pre_t1)
{
    if (self_prefix) {
        tile_prefixes(a.tsumP, tile, lds, pre_t, pre_t1);
        if (threadIdx.x == 0) a.tpreP[tile] = *pre_t;
    } else {
        *pre_t = a.tpreP[tile];
        *pre_t1 = a.tpreP[tile + 1];
    }
}

struct esa_classify_kernel {
    static constexpr int LB = CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, EsaArgs a, int self_prefix)
{
    __shared__ ChainLds sh;
    const int64_t L = *a.Lp;
    const int64_t tile = kg_.bid;
    if (tile * CTILE >= L) return;
    double v[CI], pre_t, pre_t1;
    fetch_tile(ArraySrc{a.x}, tile * CTILE, L, v);
    get_prefixes(a, tile, self_prefix, sh.d, &pre_t, &pre_t1);
    classify_tile(a, v, tile, L, *a.v0p, pre_t, pre_t1, sh);
}
};

// The sequential part: one thread walks the sensitive elements in order from the
// chain's start value, each getting fl(value before it + s x), the value before it
// being the previous one plus the regular sum in between (exact: the run stays in one
// binade).  The list is in global memory (staged through LDS in rounds) or, from the
// one-block kernel, already in LDS (lpre, lsx non-null).  A list beyond its capacity
// leaves every element after the last one kept to the repair.
__device__ void esa_walk_block(const EsaArgs &a, int64_t ns, const double *lpre, const double *lsx)
{
    __shared__ double sp[WALK_CHUNK], sx[WALK_CHUNK], sv[WALK_CHUNK];
    __shared__ double Vd;
    const int t = threadIdx.x;
    if (ns > a.smax) {
        if (t == 0)
            atomicMin((unsigned long long *)&a.first_bad[1], (unsigned long long)(a.s_idx[a.smax - 1] + 1));
        ns = a.smax;
    }
    if (lpre) {
        if (t == 0) {
            double vd = *a.v0p;
            for (int64_t k = 0; k < ns; k++) {
                const double pred = lpre[k] == 0.0 ? vd : vd + lpre[k];
                vd = pred + lsx[k];
                a.s_v[k] = vd;
            }
        }
        return;
    }
    if (t == 0) Vd = *a.v0p;
    __syncthreads();
    for (int64_t c0 = 0; c0 < ns; c0 += WALK_CHUNK) {
        const int64_t k = c0 + t;
        if (t < WALK_CHUNK && k < ns) {
            sp[t] = a.s_pre[k];
            sx[t] = a.sign * a.x[a.s_idx[k]];
        }
        __syncthreads();
        if (t == 0) {
            double vd = Vd;
            const int cnt = (int)(ns - c0 < WALK_CHUNK ? ns - c0 : WALK_CHUNK);
            for (int u = 0; u < cnt; u++) {
                const double pred = sp[u] == 0.0 ? vd : vd + sp[u];
                vd = pred + sx[u];
                sv[u] = vd;
            }
            Vd = vd;
        }
        __syncthreads();
        if (t < WALK_CHUNK && k < ns) a.s_v[k] = sv[t];
        __syncthreads();
    }
}

// The tiles' sensitive offsets and open-segment carries (a segmented scan of the tile
// aggregates), by a group of CT threads; returns the chain's total.
__device__ Seg walk_scan(const EsaArgs &a, int64_t nt, Seg *lds)
{
    const int t = threadIdx.x % CT;
    const int64_t chunk = (nt + CT - 1) / CT;
    const int64_t b0 = (int64_t)t * chunk;
    Seg tot;
    if (chunk <= WALK_REG) {
        // the thread's tile entries in registers, every load issued before the first use
        Seg v[WALK_REG];
#pragma unroll
        for (int u = 0; u < WALK_REG; u++) {
            const int64_t b = b0 + u;
            v[u] = u < chunk && b < nt ? Seg{a.ttail[b], a.tcnt[b]} : Seg{0, 0};
        }
        Seg acc{0, 0};
#pragma unroll
        for (int u = 0; u < WALK_REG; u++) acc = seg_then(acc, v[u]);
        Seg run = block_excl_seg(acc, lds, &tot);
#pragma unroll
        for (int u = 0; u < WALK_REG; u++) {
            const int64_t b = b0 + u;
            if (u < chunk && b < nt) {
                a.toff[b] = run.cnt;
                a.tcarry[b] = run.sum;
            }
            run = seg_then(run, v[u]);
        }
    } else {
        Seg acc{0, 0};
        for (int64_t b = b0; b < b0 + chunk && b < nt; b++) acc = seg_then(acc, Seg{a.ttail[b], a.tcnt[b]});
        Seg run = block_excl_seg(acc, lds, &tot);
        for (int64_t b = b0; b < b0 + chunk && b < nt; b++) {
            a.toff[b] = run.cnt;
            a.tcarry[b] = run.sum;
            run = seg_then(run, Seg{a.ttail[b], a.tcnt[b]});
        }
    }
    if (t == 0) *a.s_n = tot.cnt;
    __syncthreads();                                // (also makes the block's global writes visible to it)
    return tot;
}

// LDS of the walk: the appended list put in order
struct WalkLds {
    Seg s[CT / 64];
    double pre[RAW_CAP], sx[RAW_CAP];
};

// The appended list (ns entries) put in order, by a group of CT threads: an element's place is
// its tile's offset and its number there.
__device__ void walk_list(const EsaArgs &a, int64_t ns, double *pre, double *sx)
{
    for (int64_t e = threadIdx.x % CT; e < ns; e += CT) {
        const int64_t j = a.raw_idx[e], tile = j / CTILE;
        const int32_t k = a.raw_bp[a.raw_cap + e];
        const int64_t at = a.toff[tile] + k;
        if (a.s_idx) a.s_idx[at] = j;
        pre[at] = seg_value(a.raw_part[e] + (k == 0 ? a.tcarry[tile] : 0), a.raw_bp[e]);
        sx[at] = a.raw_sx[e];
    }
    __syncthreads();
}

// One block: the scan, then the ordered list of the sensitive elements and the walk.  The
// list is the classification's appended one when it holds every sensitive element;
// otherwise (more than RAW_CAP, never for an ordinary cluster) this block classifies the
// tiles again one after another and lists them in order, slowly but exactly.
struct esa_walk_kernel {
    static constexpr int LB = CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, EsaArgs a)
{
    __shared__ WalkLds sh;
    const int t = threadIdx.x;
    const int64_t L = *a.Lp;
    const int64_t nt = (L + CTILE - 1) / CTILE;
    const Seg tot = walk_scan(a, nt, sh.s);
    const int64_t ns = tot.cnt;
    if (ns > RAW_CAP) {
        __shared__ double ldsd[CT / 64];
        __shared__ double tbuf[TILE_LDS];
        for (int64_t tile = 0; tile < nt; tile++) {
            TileItems it;
            double v[CI];
            fetch_tile(ArraySrc{a.x}, tile * CTILE, L, v);
            tile_classify(a, v, tile, L, *a.v0p, it, ldsd, tbuf, a.tpreP[tile], a.tpreP[tile + 1]);
            Seg ttot;
            const Seg pre = block_excl_seg(items_seg(it), sh.s, &ttot);
            int64_t k = a.toff[tile] + pre.cnt;
            int64_t cur = pre.sum + (pre.cnt ? 0 : a.tcarry[tile]);
            const int64_t j0 = tile * CTILE + (int64_t)t * CI;
            for (int u = 0; u < CI; u++) {
                if ((it.sens >> u) & 1) {
                    if (k < a.smax) {
                        a.s_idx[k] = j0 + u;
                        a.s_pre[k] = seg_value(cur, it.bp[u]);
                    }
                    k++;
                    cur = 0;
                } else {
                    cur += it.R[u];
                }
            }
            __syncthreads();
        }
        esa_walk_block(a, ns, nullptr, nullptr);
        return;
    }
    walk_list(a, ns, sh.pre, sh.sx);
    esa_walk_block(a, ns, sh.pre, sh.sx);
}
};

// Parallel rebuild of one tile from the last sensitive value before every element, and
// verification of the recurrence against the values rebuilt (the value before a tile is
// rebuilt exactly as the previous tile's block rebuilds it).  vc: the start value that
// the classification used, v0: the exact one.  nv: the thread's values; *before: the
// value before its first element.  Returns the thread's first violation, or L.
// s_v: the values of the ns_eff listed sensitive elements.
__device__ __forceinline__ int64_t rebuild_tile(const EsaArgs &a, const double (&v)[CI], int64_t tile, int64_t L, double vc,
                                                double v0, const double *s_v, int64_t ns_eff, ChainLds &sh, TileItems &it,
                                                double (&nv)[CI], double *before)
{
    const int64_t base = tile * CTILE;
    const int t = threadIdx.x;
    const int64_t toff = a.toff[tile], tcarry = a.tcarry[tile];
    tile_classify(a, v, tile, L, vc, it, sh.d, sh.tbuf, a.tpreP[tile], a.tpreP[tile + 1]);
    Seg tot;
    const Seg pre = block_excl_seg(items_seg(it), sh.s, &tot);
    int64_t k = toff + pre.cnt;                       // rank of the next sensitive element
    int64_t cur = pre.sum + (pre.cnt ? 0 : tcarry);
    const int64_t j0 = base + (int64_t)t * CI;
#pragma unroll
    for (int u = 0; u < CI; u++) {
        if ((it.sens >> u) & 1) {
            nv[u] = k < ns_eff ? s_v[k] : it.pa[u];
            k++;
            cur = 0;
        } else {
            cur += it.R[u];
            const int64_t kk = k - 1;                 // the last sensitive element before
            if (kk >= ns_eff) {
                nv[u] = it.pa[u];
            } else {
                const double b = kk >= 0 ? s_v[kk] : v0;
                nv[u] = cur == 0 ? b : b + seg_value(cur, it.bp[u]);
            }
        }
    }
    sh.lastv[t] = nv[CI - 1];
    __syncthreads();
    double prev;
    if (t > 0) {
        prev = sh.lastv[t - 1];
    } else if (tile == 0) {
        prev = v0;
    } else {
        const int64_t kk = toff - 1;
        if (kk >= ns_eff) prev = it.pa[0] - it.sx[0];        // past the list: already left to the repair
        else if (kk >= 0 && a.s_idx[kk] == base - 1) prev = s_v[kk];
        else {
            const double b = kk >= 0 ? s_v[kk] : v0;
            // (a tile past the chain's end classifies nothing: its run has the binade of b)
            prev = tcarry == 0 ? b : b + seg_value(tcarry, base < L ? it.bp[0] : binade_of(b));
        }
    }
    *before = prev;
    int64_t bad = L;
#pragma unroll
    for (int u = 0; u < CI; u++) {
        const int64_t j = j0 + u;
        if (j < L) {
            const double want = prev + it.sx[u];
            if (want != nv[u] && j < bad) bad = j;
        }
        prev = nv[u];
    }
    return bad;
}

struct esa_rebuild_kernel {
    static constexpr int LB = CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, EsaArgs a)
{
    __shared__ ChainLds sh;
    const int64_t L = *a.Lp;
    const int64_t tile = kg_.bid;
    if (tile * CTILE >= L) return;
    const double v0 = *a.v0p;
    TileItems it;
    double v[CI], nv[CI], before;
    fetch_tile(ArraySrc{a.x}, tile * CTILE, L, v);
    const int64_t ns = *a.s_n;
    const int64_t bad = rebuild_tile(a, v, tile, L, v0, v0, a.s_v, ns < a.smax ? ns : a.smax, sh, it, nv, &before);
    if (bad < L) atomicMin((unsigned long long *)&a.first_bad[1], (unsigned long long)bad);
    store_tile(a.g, tile * CTILE, L, sh.tbuf, nv);
}
};

// The repair, only after a violation (the estimate's bound or the list's capacity
// exceeded, which a monotone chain of ordinary size never does): the recurrence
// itself from the first violating element on, one thread over chunks that the block
// stages through LDS in coalesced rows.
constexpr int FIN_CHUNK = 4 * WALK_T;
struct chain_finish_kernel {
    static constexpr int LB = WALK_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, EsaArgs a)
{
    __shared__ double buf[FIN_CHUNK];
    __shared__ double vlast;
    const int64_t L = *a.Lp;
    const int64_t j0 = a.first_bad[1];
    if (j0 >= L) return;
    const int t = threadIdx.x;
    if (t == 0) vlast = j0 == 0 ? *a.v0p : a.g[j0 - 1];
    for (int64_t c0 = j0; c0 < L; c0 += FIN_CHUNK) {
        const int cnt = (int)(L - c0 < FIN_CHUNK ? L - c0 : FIN_CHUNK);
        for (int i = t; i < cnt; i += WALK_T) buf[i] = a.sign * a.x[c0 + i];
        __syncthreads();
        if (t == 0) {
            double v = vlast;
            for (int i = 0; i < cnt; i++) {
                v = v + buf[i];
                buf[i] = v;
            }
            vlast = v;
        }
        __syncthreads();
        for (int i = t; i < cnt; i += WALK_T) a.g[c0 + i] = buf[i];
        __syncthreads();
    }
}
};

// ---------------------------------------------------------------- the three chains
struct pot_init_kernel { static constexpr int LB = 1024, MB = 0; static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s) { s->first_inf = s->n_max + 1; } };

// cmc_utils.c:685-696: the count stops at the first k with !(r[k] < SF_INFINITY).
struct pot_count_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ r, DevScalars *s)
{
    int64_t k = 1 + (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (k > s->n_max) return;
    if (!(r[k] < CMCG_SF_INFINITY)) atomicMin((unsigned long long *)&s->first_inf, (unsigned long long)k);
}
};

// The three chains of the potential.  A and B are classified together: chain B starts
// from the total mass, whose estimate (the tile sums of A) is good enough to tell the
// binades (EsaArgs::extra), so B need not wait for A's walk; one block then walks A and B.
// Chain A needs only its last value, so it is never rebuilt: for masses that are not
// negative the bound on the estimate is rigorous, and any other mass takes the repair.
// B's rebuild forms chain C's increments at once (M_k is not stored), and C's rebuild
// writes the potential and the node tables.  Eight launches; each chain by itself took
// five, and the counts and copies five more.  The phase: 0.109 -> 0.070 ms at N = 1e4, where
// a launch costs 4 to 5 us whatever it does, 0.128 -> 0.090 at 1e6, 0.242 -> 0.179 at 4e6
// (there the passes over memory bound it: 42, 41 and 34 us for the A and B classification
// and the two rebuilds).
struct PotArgs {
    const double *m;
    double *r, *phi;
    DevScalars *s;
    double nstar;
    double *xc;                 // chain C's increments
    double *scal;               // [0] 0.0 (C's start), [1] Mtotal (B's start), [2] its estimate
    // nonzero: the chains go through the repair.  A kernel reads only the words that earlier
    // kernels set: [0] classification of A and B, [1] rebuild of B, [2] rebuild of C
    int64_t *flag;
    double2 *nodes;             // packed (r, phi) of every node
    int counted;                // N_MAX from the count of radii below SF_INFINITY (pot_count_kernel)
    EsaArgs a, b, c;
    __device__ __forceinline__ int64_t lb(int64_t n) const { return n > 1 ? n - 1 : 0; }
    __device__ __forceinline__ bool flagged(int words) const
    {
        int64_t any = 0;
        for (int q = 0; q < words; q++) any |= flag[q];
        return any != 0;
    }
};
struct SrcA {
    const double *__restrict__ m;
    __device__ __forceinline__ double operator()(int64_t j) const { return m[1 + j]; }
};
// star_m[k] / clus.N_STAR, k = N - j
struct SrcB {
    const double *__restrict__ m;
    int64_t n;
    double nstar;
    __device__ __forceinline__ double operator()(int64_t j) const { return m[n - j] / nstar; }
};

// the total mass from chain A's last value (cmc_utils.c:703)
__device__ __forceinline__ double pot_mass(const KParams &P, double mprev) { return mprev * P.madhoc + P.cenma_m * P.madhoc; }

// The tile sums of A and B, N_MAX and the sentinels (cmc_utils.c:713-714), the chains'
// flags and lists cleared.
struct pot_sums_kernel {
    static constexpr int LB = CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, PotArgs p)
{
    __shared__ double lds[CT / 64];
    const int64_t n = p.counted ? p.s->first_inf - 1 : p.s->n_max;
    const int64_t base = (int64_t)kg_.bid * CTILE;
    if (kg_.bid == 0 && threadIdx.x == 0) {
        if (p.counted) p.s->n_max = n;               // the other blocks read first_inf
        p.scal[0] = 0.0;
        for (int q = 0; q < 3; q++) p.flag[q] = 0;
        *p.a.raw_n = 0;
        *p.b.raw_n = 0;
        *p.c.raw_n = 0;
        p.r[n + 1] = CMCG_SF_INFINITY;
        p.phi[n + 1] = 0.0;
    }
    const SrcA sa{p.m};
    const SrcB sb{p.m, n, p.nstar};
    double va[CI], vb[CI];
#pragma unroll
    for (int u = 0; u < CI; u++) {
        const int64_t j = base + u * CT + threadIdx.x;
        va[u] = j < n ? sa(j) : 0.0;
        vb[u] = j < p.lb(n) ? sb(j) : 0.0;
    }
    double ta = 0.0, tb = 0.0;
#pragma unroll
    for (int u = 0; u < CI; u++) { ta += va[u]; tb -= vb[u]; }
    ta = tree_sum(ta, lds);
    tb = tree_sum(tb, lds);
    if (threadIdx.x == 0) {
        p.a.tsumP[kg_.bid] = ta;
        p.b.tsumP[kg_.bid] = tb;
    }
}
};

// Blocks 0 .. tiles - 1 classify chain A's tiles, the rest chain B's.
struct pot_classify_ab_kernel {
    static constexpr int LB = CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, PotArgs p, KParams P, int self_prefix)
{
    __shared__ ChainLds sh;
    const int64_t n = p.s->n_max, nt = kg_.nb / 2;
    const bool isb = kg_.bid >= nt;
    const int64_t tile = isb ? kg_.bid - nt : kg_.bid;
    if (tile * CTILE >= n) return;
    double v[CI], pre_t, pre_t1;
    if (isb) fetch_tile(SrcB{p.m, n, p.nstar}, tile * CTILE, p.lb(n), v);
    else fetch_tile(SrcA{p.m}, tile * CTILE, n, v);
    // the total mass as chain A's sums estimate it, by the same sums in every block of B
    const int64_t live = (n + CTILE - 1) / CTILE;
    double est = 0.0;
    if (isb)
        for (int64_t q = threadIdx.x; q < live; q += CT) est += p.a.tsumP[q];
    get_prefixes(isb ? p.b : p.a, tile, self_prefix, sh.d, &pre_t, &pre_t1);
    bool ok;
    if (isb) {
        est = pot_mass(P, tree_sum(est, sh.d));
        if (tile == 0 && threadIdx.x == 0) p.scal[2] = est;
        EsaArgs b = p.b;
        b.extra = n;
        ok = classify_tile(b, v, tile, p.lb(n), est, pre_t, pre_t1, sh);
    } else {
        ok = classify_tile(p.a, v, tile, n, 0.0, pre_t, pre_t1, sh);
    }
    if (!ok) p.flag[0] = 1;
}
};

__device__ __forceinline__ double lane_value(double x, int lane)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, lane), hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), lane);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The walk over ns listed elements from v, by one whole wave: 64 elements at a time in
// its lanes' registers, so that the chain of additions waits on no memory.  s_v (which may
// be pre or sx) receives the value after each element; every lane returns the last.  (Adding a
// run of nothing, 0.0, changes no value that is not -0.0, and the chains hold none.)
__device__ __forceinline__ double pot_walk(int64_t ns, double v, const double *pre, const double *sx, double *s_v)
{
    const int lane = threadIdx.x & 63;
    double np = lane < ns ? pre[lane] : 0.0, nx = lane < ns ? sx[lane] : 0.0;
    for (int64_t c = 0; c < ns; c += 64) {
        const int cnt = (int)(ns - c < 64 ? ns - c : 64);
        const double p = np, x = nx;
        if (c + 64 + lane < ns) {                     // the next 64, while these are walked
            np = pre[c + 64 + lane];
            nx = sx[c + 64 + lane];
        }
        double mine = 0.0;
        auto step = [&](int k) {
            v = (v + lane_value(p, k)) + lane_value(x, k);
            if (lane == k) mine = v;
        };
        if (cnt == 64) {
#pragma unroll 16
            for (int k = 0; k < 64; k++) step(k);
        } else {
            for (int k = 0; k < cnt; k++) step(k);
        }
        if (lane < cnt) s_v[c + lane] = mine;
    }
    return v;
}

// after chain A: Mtotal, Rtidal (cmc_utils.c:703-707), NaN check (:688-691)
__device__ __forceinline__ void pot_total(const PotArgs &p, const KParams &P, double mprev)
{
    DevScalars *s = p.s;
    if (isnan(mprev)) dev_set_error(s, CMCG_E_NAN, s->n_max);
    const double Mtotal = pot_mass(P, mprev);
    s->Mtotal = Mtotal;
    s->Rtidal = P.orbit_r * pow(Mtotal, 1.0 / 3.0);
    p.scal[1] = Mtotal;
}

// Chains A and B: half the block puts each list in order, then one wave walks A, finishes
// the total mass and walks B from it.  (Block by block, B's list after A's walk: 21 us at
// N = 4e6 instead of 17; B walked again by every block of its rebuild: no faster in all.)
struct pot_walk_ab_kernel {
    static constexpr int LB = 2 * CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, PotArgs p, KParams P)
{
    __shared__ WalkLds sh[2];
    __shared__ Seg tot[2];
    const int64_t n = p.s->n_max, nt = (n + CTILE - 1) / CTILE;
    if (p.flag[0]) return;                            // the repair runs the chains itself
    const int h = threadIdx.x / CT;
    const EsaArgs &c = h ? p.b : p.a;
    const Seg mine = walk_scan(c, nt, sh[h].s);
    if (threadIdx.x % CT == 0) tot[h] = mine;
    __syncthreads();
    // lists longer than LDS holds go through memory, one after the other
    const bool lds = tot[0].cnt <= RAW_CAP && tot[1].cnt <= RAW_CAP;
    double *pa = lds ? sh[0].pre : p.b.s_pre, *xa = lds ? sh[0].sx : p.b.s_v;
    double *pb = lds ? sh[1].pre : p.b.s_pre, *xb = lds ? sh[1].sx : p.b.s_v;
    if (lds) walk_list(c, mine.cnt, h ? pb : pa, h ? xb : xa);
    else walk_list(p.a, h ? 0 : tot[0].cnt, pa, xa);
    double v = 0.0;                                   // chain A's last value (wave 0)
    if (threadIdx.x < 64) {
        v = pot_walk(tot[0].cnt, 0.0, pa, xa, xa);
        if (tot[0].sum != 0) v += seg_value(tot[0].sum, binade_of(v));   // the run after the last stays in one binade
        if (threadIdx.x == 0) pot_total(p, P, v);
    }
    if (!lds) {
        __syncthreads();
        walk_list(p.b, h ? tot[1].cnt : 0, pb, xb);
    }
    if (threadIdx.x < 64) pot_walk(tot[1].cnt, pot_mass(P, v), pb, xb, p.b.s_v);
}
};

// Chain B rebuilt and verified; from the enclosed masses chain C's increments
// p_k = M_k * (1/r_k - 1/r_{k+1}), k = N - j, with the reference's roundings, and their
// tile sums; chain C runs on w = -phi, w_k = fl(w_{k+1} + p_k).  M_k is the value before
// B's element j.
struct pot_rebuild_b_kernel {
    static constexpr int LB = CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, PotArgs p)
{
    __shared__ ChainLds sh;
    const int64_t n = p.s->n_max;
    const int64_t tile = kg_.bid, base = tile * CTILE;
    const int t = threadIdx.x;
    if (base >= n || p.flag[0]) return;
    EsaArgs b = p.b;
    b.extra = n;
    const int64_t lb = p.lb(n);
    double v[CI], rk[CI], rk1[CI];
    fetch_tile(SrcB{p.m, n, p.nstar}, base, lb, v);
#pragma unroll
    for (int u = 0; u < CI; u++) {
        const int64_t j = base + u * CT + t;
        rk[u] = j < n ? p.r[n - j] : 1.0;
        rk1[u] = j < n ? p.r[n - j + 1] : 1.0;
    }
    TileItems it;
    double nv[CI], before;
    const int64_t bad = rebuild_tile(b, v, tile, lb, p.scal[2], p.scal[1], b.s_v, *b.s_n, sh, it, nv, &before);
    if (bad < lb) p.flag[1] = 1;
    // 1/r_k - 1/r_{k+1} of the tile through LDS
    __syncthreads();                                  // tbuf free
#pragma unroll
    for (int u = 0; u < CI; u++) sh.tbuf[tile_slot(u * CT + t)] = 1.0 / rk[u] - 1.0 / rk1[u];
    __syncthreads();
    double x[CI], acc = 0.0;
#pragma unroll
    for (int u = 0; u < CI; u++) {
        x[u] = (u == 0 ? before : nv[u > 0 ? u - 1 : 0]) * sh.tbuf[tile_slot(t * CI + u)];
        if (base + (int64_t)t * CI + u < n) acc += x[u];
    }
    const double tot = tree_sum(acc, sh.d);           // (a barrier: every thread is past its reads of tbuf)
    if (t == 0) p.c.tsumP[tile] = tot;
    store_tile(p.xc, base, n, sh.tbuf, x);
}
};

struct pot_classify_c_kernel {
    static constexpr int LB = CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, PotArgs p, int self_prefix)
{
    __shared__ ChainLds sh;
    const int64_t n = p.s->n_max, tile = kg_.bid;
    if (tile * CTILE >= n || p.flagged(2)) return;
    double v[CI], pre_t, pre_t1;
    fetch_tile(ArraySrc{p.xc}, tile * CTILE, n, v);
    get_prefixes(p.c, tile, self_prefix, sh.d, &pre_t, &pre_t1);
    classify_tile(p.c, v, tile, n, 0.0, pre_t, pre_t1, sh);
}
};

struct pot_walk_c_kernel {
    static constexpr int LB = CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, PotArgs p)
{
    __shared__ WalkLds sh;
    if (p.flagged(2)) return;
    Seg tot;
    tot = walk_scan(p.c, (p.s->n_max + CTILE - 1) / CTILE, sh.s);
    const bool lds = tot.cnt <= RAW_CAP;
    double *pre = lds ? sh.pre : p.c.s_pre, *sx = lds ? sh.sx : p.c.s_v;
    walk_list(p.c, tot.cnt, pre, sx);
    if (threadIdx.x < 64) pot_walk(tot.cnt, 0.0, pre, sx, p.c.s_v);
}
};

// phi_k into the potential and the node tables, which the searches of set_velocities3 and
// the orbit phase read
__device__ __forceinline__ void put_node(const PotArgs &p, int64_t k, double r, double phi)
{
    p.nodes[k] = make_double2(r, phi);
}
// nodes 0 (cmc_utils.c:729; phi1 = phi[1], the sentinel's 0 when there are no stars) and n + 1
__device__ __forceinline__ void put_ends(const PotArgs &p, const KParams &P, int64_t n, double phi1)
{
    const double p0 = phi1 + P.cenma_m * P.madhoc / p.r[1];
    p.phi[0] = p0;
    put_node(p, 0, p.r[0], p0);
    put_node(p, n + 1, CMCG_SF_INFINITY, 0.0);
}

// Chain C rebuilt and verified, phi_k = -w_k, k = N - j, and the node tables.
struct pot_rebuild_c_kernel {
    static constexpr int LB = CT, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, PotArgs p, KParams P)
{
    __shared__ ChainLds sh;
    const int64_t n = p.s->n_max;
    const int64_t tile = kg_.bid, base = tile * CTILE;
    const int t = threadIdx.x;
    if (p.flagged(2)) return;
    if (n == 0 && kg_.bid == 0 && t == 0) put_ends(p, P, n, 0.0);
    if (base >= n) return;
    TileItems it;
    double v[CI], rk[CI], nv[CI], before;
    fetch_tile(ArraySrc{p.xc}, base, n, v);
#pragma unroll
    for (int u = 0; u < CI; u++) {
        const int64_t j = base + u * CT + t;
        rk[u] = j < n ? p.r[n - j] : 1.0;
    }
    const int64_t bad = rebuild_tile(p.c, v, tile, n, 0.0, 0.0, p.c.s_v, *p.c.s_n, sh, it, nv, &before);
    if (bad < n) p.flag[2] = 1;
    __syncthreads();                                  // tbuf free
#pragma unroll
    for (int u = 0; u < CI; u++) sh.tbuf[tile_slot(t * CI + u)] = nv[u];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < CI; u++) {
        const int i = u * CT + t;
        const int64_t k = n - (base + i);
        if (k < 1) break;
        const double ph = -sh.tbuf[tile_slot(i)];
        p.phi[k] = ph;
        if (isnan(ph)) dev_set_error(p.s, CMCG_E_NAN, k);
        put_node(p, k, rk[u], ph);
        if (k == 1) put_ends(p, P, n, ph);
    }
}
};

// The repair (a mass below zero, infinite or NaN, a violated recurrence: never an ordinary
// cluster; the test hook forces it): the three recurrences
// themselves, one thread over chunks that the block stages through LDS.
constexpr int FIX_CHUNK = 2 * WALK_T;
struct pot_finish_kernel {
    static constexpr int LB = WALK_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, PotArgs p, KParams P)
{
    __shared__ double x[FIX_CHUNK], y[FIX_CHUNK];
    __shared__ double va, vm;
    if (!p.flagged(3)) return;
    const int64_t n = p.s->n_max;
    const int t = threadIdx.x;
    if (t == 0) va = 0.0;
    for (int64_t c = 0; c < n; c += FIX_CHUNK) {
        const int cnt = (int)(n - c < FIX_CHUNK ? n - c : FIX_CHUNK);
        for (int i = t; i < cnt; i += WALK_T) x[i] = p.m[1 + c + i];
        __syncthreads();
        if (t == 0) {
            double v = va;
            for (int i = 0; i < cnt; i++) v = v + x[i];
            va = v;
        }
        __syncthreads();
    }
    if (t == 0) {
        pot_total(p, P, va);
        vm = p.scal[1];
        va = 0.0;
    }
    for (int64_t c = 0; c < n; c += FIX_CHUNK) {
        const int cnt = (int)(n - c < FIX_CHUNK ? n - c : FIX_CHUNK);
        for (int i = t; i < cnt; i += WALK_T) {
            const int64_t k = n - (c + i);
            x[i] = p.m[k] / p.nstar;
            y[i] = 1.0 / p.r[k] - 1.0 / p.r[k + 1];
        }
        __syncthreads();
        if (t == 0) {
            double M = vm, w = va;
            for (int i = 0; i < cnt; i++) {
                w = w + M * y[i];
                M = M - x[i];
                y[i] = w;
            }
            vm = M;
            va = w;
        }
        __syncthreads();
        for (int i = t; i < cnt; i += WALK_T) {
            const int64_t k = n - (c + i);
            const double ph = -y[i];
            p.phi[k] = ph;
            if (isnan(ph)) dev_set_error(p.s, CMCG_E_NAN, k);
            put_node(p, k, p.r[k], ph);
        }
        __syncthreads();
    }
    if (t == 0) put_ends(p, P, n, n > 0 ? -va : 0.0);
}
};

struct pot_at_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ r, const double *__restrict__ phi, DevScalars *s,
                              const double *__restrict__ x, double *__restrict__ out, int64_t count)
{
    int64_t i = (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    if (i >= count) return;
    int64_t n = s->n_max;
    bool bad = false;
    double v = potential_at(r, phi, n, x[i], 1, n + 1, &bad);
    if (bad) { dev_set_error(s, CMCG_E_BRACKET, i); v = 0.0; }
    out[i] = v;
}
};

// Independent chains side by side: the buffers of chain c lie c words (xs for the increments
// and values) after those of chain 0.
__device__ __forceinline__ EsaArgs esa_chain(EsaArgs e, int64_t c, int64_t words, int64_t xs)
{
    const int64_t w = c * words;
    e.x += c * xs; e.g += c * xs;
    e.v0p += w; e.first_bad += w; e.Lp += w;
    e.tsumP += w; e.tpreP += w; e.tcnt += w; e.ttail += w; e.toff += w; e.tcarry += w;
    e.s_idx += w; e.s_pre += w; e.s_v += w; e.s_n += w;
    e.raw_n += w; e.raw_idx += w; e.raw_part += w; e.raw_bp += 2 * w; e.raw_sx += w;
    return e;
}
// kernel K of every chain in one launch, `per` blocks each
template <class K>
struct esa_each {
    static constexpr int LB = K::LB, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, EsaArgs e, int64_t words, int64_t xs, unsigned per)
    {
        const unsigned c = kg_.bid / per;
        K::run(KGrid{kg_.bid - c * per, per, 0, 1}, esa_chain(e, c, words, xs));
    }
};
template <class K>
struct esa_each1 {
    static constexpr int LB = K::LB, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, EsaArgs e, int64_t words, int64_t xs, unsigned per, int64_t arg)
    {
        const unsigned c = kg_.bid / per;
        K::run(KGrid{kg_.bid - c * per, per, 0, 1}, esa_chain(e, c, words, xs), arg);
    }
};

// The increments must be in every chain's x.  (One after another, the five chains of
// comp_mass_percent and the seven of central_calculate took 30 and 50 launches, each too
// small to fill the chip: 380 and 350 us at N = 1e6.)
hipError_t run_chains(const EsaArgs &e, int64_t words, int64_t xs, int chains, int64_t n_ub, hipStream_t st)
{
    int64_t ntiles = (n_ub + CTILE - 1) / CTILE;
    if (ntiles < 1) ntiles = 1;
    const unsigned per = (unsigned)ntiles;
    const dim3 gt(per * chains), gc((unsigned)chains), bt(CT);
    kl<esa_each<esa_sum_kernel>>(gt, bt, 0, st, e, words, xs, per);
    const bool self_prefix = ntiles <= SELF_PREFIX_MAX;
    if (!self_prefix) kl<esa_each1<esa_tile_scan_kernel>>(gc, dim3(WALK_T), 0, st, e, words, xs, 1u, ntiles);
    kl<esa_each1<esa_classify_kernel>>(gt, bt, 0, st, e, words, xs, per, (int64_t)self_prefix);
    kl<esa_each<esa_walk_kernel>>(gc, bt, 0, st, e, words, xs, 1u);
    kl<esa_each<esa_rebuild_kernel>>(gt, bt, 0, st, e, words, xs, per);
    kl<esa_each<chain_finish_kernel>>(gc, dim3(WALK_T), 0, st, e, words, xs, 1u);
    return hipGetLastError();
}

// The buffers of up to REPORT_CHAINS chains: the lists and tile sums in the report workspace,
// the increments and values in the sort's record scratch (16 words per star, free between
// sorts; 12 are used).
constexpr int REPORT_CHAINS = 6;
constexpr int64_t REPORT_LIST = 1 << 16;
int64_t report_words(int64_t T) { return 6 * T + 3 * REPORT_LIST + 8 + 4 * RAW_CAP; }
EsaArgs report_chain0(const Scratch &sc, int slack, void *work, int64_t xs)
{
    const int64_t T = sc.max_tiles;
    double *w = (double *)work;
    EsaArgs e{};
    e.slack = slack;
    e.sign = 1.0;
    e.x = (const double *)sc.sort_aos;
    e.g = (double *)sc.sort_aos + REPORT_CHAINS * xs;
    e.tsumP = w;
    e.tpreP = w + T;
    e.tcnt = (int64_t *)(w + 2 * T);
    e.ttail = (int64_t *)(w + 3 * T);
    e.toff = (int64_t *)(w + 4 * T);
    e.tcarry = (int64_t *)(w + 5 * T);
    w += 6 * T;
    e.s_idx = (int64_t *)w;
    e.s_pre = w + REPORT_LIST;
    e.s_v = w + 2 * REPORT_LIST;
    e.smax = REPORT_LIST;
    w += 3 * REPORT_LIST;
    e.s_n = (int64_t *)w;
    e.raw_n = (int64_t *)(w + 1);
    e.first_bad = (int64_t *)(w + 2);
    e.Lp = (const int64_t *)(w + 4);
    e.v0p = w + 5;
    w += 8;
    e.raw_idx = (int64_t *)w;
    e.raw_part = (int64_t *)(w + RAW_CAP);
    e.raw_bp = (int32_t *)(e.raw_part + RAW_CAP);
    e.raw_sx = (double *)(e.raw_part + 2 * RAW_CAP);
    e.raw_cap = RAW_CAP;
    return e;
}

// The chains' per-tile buffers in the context's scratch (tile_sums: six 8-byte words per tile),
// their lists, of as many elements as there are stars, in the sort's records (free between
// sorts: 11 of their 16 words a star).
// set: 0 or 1, for two chains that are classified together
EsaArgs esa_args(const Scratch &sc, int slack, int set = 0)
{
    const int64_t T = sc.max_tiles;
    double *tb = sc.tile_sums + 6 * T * set;
    EsaArgs e{};
    e.slack = slack;
    e.tsumP = tb;
    e.tpreP = tb + T;
    e.tcnt = (int64_t *)(tb + 2 * T);
    e.ttail = (int64_t *)(tb + 3 * T);
    e.toff = (int64_t *)(tb + 4 * T);
    e.tcarry = (int64_t *)(tb + 5 * T);
    e.s_n = sc.esa_n;
    e.raw_n = sc.esa_n + 1 + set;
    const int64_t cap = sc.sort_aos_cap;
    double *w = (double *)sc.sort_aos;
    e.smax = e.raw_cap = cap;
    e.s_idx = (int64_t *)w;
    e.s_pre = w + cap;
    e.s_v = w + 2 * cap;
    w += (3 + 4 * set) * cap;
    e.raw_idx = (int64_t *)w;
    e.raw_part = (int64_t *)(w + cap);
    e.raw_bp = (int32_t *)(w + 2 * cap);
    e.raw_sx = w + 3 * cap;
    return e;
}
} // namespace

// ---------------------------------------------------------------- comp_mass_percent
// cmc_utils.c:872-982 for one rank.  Chain M: mprev_k = mprev_{k-1} + m_k / N_STAR
// (k = 1..N_MAX, from cenma.m madhoc or 0); chains T_r, T_t, V_r, V_t: the running
// sums of 0.5 m madhoc vr vr, 0.5 m madhoc vt vt, vr vr, vt vt (k = 1..N_MAX_NEW).
// Each is the reference's sequential recurrence, solved by the same exact emulation
// as the potential's chains.
constexpr int MPC_MAX = 256;
struct MassPcOut {
    double v[8][MPC_MAX];        // mass_r, ave_mass_r, densities_r, ke_rad, ke_tan, v2_rad, v2_tan, (unused)
    int64_t k[MPC_MAX];          // no_star_r (the index k)
    int64_t reached;             // fractions assigned
    int64_t negative;            // a mass is below zero (or NaN): the enclosed mass is not monotone
};

// Chain 0: star_m[k] / clus.N_STAR; 1 to 4: 0.5 m madhoc vr vr, 0.5 m madhoc vt vt, vr vr,
// vt vt (left to right), k = j + 1; and the chains' lengths and start values.
struct mpc_prep_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const DevFields f, const DevScalars *s, double nstar, double madhoc,
                                  double mprev0, EsaArgs e, int64_t words, int64_t xs, MassPcOut *o)
{
    const int64_t j = (int64_t)kg_.bid * blockDim.x + threadIdx.x, k = j + 1;
    const int64_t n = s->n_max, nn = s->n_max_new;
    double *x = const_cast<double *>(e.x);
    if (j < 5) {
        const_cast<int64_t *>(e.Lp)[j * words] = j == 0 ? n : nn;
        const_cast<double *>(e.v0p)[j * words] = j == 0 ? mprev0 : 0.0;
    }
    if (j < n) {
        const double m = f.m[k];
        x[j] = m / nstar;
        if (!(m >= 0.0)) o->negative = 1;
    }
    if (j < nn) {
        const double m = f.m[k], vr = f.vr[k], vt = f.vt[k];
        x[xs + j] = 0.5 * m * madhoc * vr * vr;
        x[2 * xs + j] = 0.5 * m * madhoc * vt * vt;
        x[3 * xs + j] = vr * vr;
        x[4 * xs + j] = vt * vt;
    }
}
};

// x^3 from x*x exactly as a double-double, times x: within 2^-50 ulp of the correctly
// rounded cube (pow(x, 3) of a correctly rounding libm)
__device__ __forceinline__ double cube_rn(double x)
{
    const double p = x * x, e = __builtin_fma(x, x, -p);
    const double q = p * x, f1 = __builtin_fma(p, x, -q);
    return q + (f1 + e * x);
}

// The fractions' indices (one fraction per star at most, as the reference's loop) from the
// enclosed-mass chain g[k-1] = mprev after star k, which does not decrease: a thread finds
// each fraction's first k with g[k-1] > pc Mtotal, one thread then moves them past the
// fraction before, and the threads take the values there.  With a negative mass it may decrease,
// and the block looks at every star after the one before.  (One thread searching for one
// fraction after another waited on 20 loads for each.)
struct mpc_finish_kernel {
    static constexpr int LB = MPC_MAX, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ r, const DevScalars *s,
                                  const double *__restrict__ g, int64_t xs, const double *__restrict__ pc, int count,
                                  int bh_include, double mprev0, double itm, double minimum_r, MassPcOut *o)
{
    __shared__ int64_t ks[MPC_MAX];
    __shared__ int reached;
    const double PI = 3.14159265358979323;                  // include/cmc/cmc.h:62
    const double Mtotal = s->Mtotal;
    const int64_t n = s->n_max;
    const int i = threadIdx.x;
    if (i < count) {
        const double thr = pc[i] * Mtotal;
        int64_t lo = 1, hi = n + 1;
        while (lo < hi) {
            const int64_t mid = lo + (hi - lo) / 2;
            if (g[mid - 1] > thr) hi = mid;
            else lo = mid + 1;
        }
        ks[i] = lo;
    }
    __syncthreads();
    if (i == 0) {
        int mc = 0;
        if (bh_include)
            for (; mc < count && mprev0 / Mtotal > pc[mc]; mc++) ks[mc] = 0;
        int64_t kprev = 0;
        for (; mc < count && !o->negative; mc++) {
            const int64_t k = ks[mc] > kprev ? ks[mc] : kprev + 1;
            if (k > n) break;
            ks[mc] = kprev = k;
        }
        reached = mc;
    }
    __syncthreads();
    if (o->negative) {
        __shared__ int64_t found;
        int64_t k = 0;
        for (int mc = reached; mc < count; mc++) {
            const double thr = pc[mc] * Mtotal;
            if (i == 0) found = n + 1;
            __syncthreads();
            for (k++; k <= n; k += MPC_MAX) {
                if (k + i <= n && g[k + i - 1] > thr) atomicMin((unsigned long long *)&found, (unsigned long long)(k + i));
                __syncthreads();
                const bool hit = found <= n;
                __syncthreads();                           // before the next round's stores
                if (hit) break;
            }
            if (found > n) break;
            k = found;
            if (i == 0) {
                ks[mc] = k;
                reached = mc + 1;
            }
            __syncthreads();
        }
    }
    if (i == 0) o->reached = reached;
    if (i >= reached) return;
    const int64_t k = ks[i];
    o->k[i] = k;
    if (k > 0) {
        const double mprev = g[k - 1];
        o->v[0][i] = r[k];
        o->v[1][i] = mprev / Mtotal / k * itm;
        o->v[2][i] = mprev / (4.0 / 3.0 * PI * cube_rn(r[k]));
        for (int t = 0; t < 4; t++) o->v[3 + t][i] = g[(t + 1) * xs + k - 1];
    } else {                                                // the central mass alone
        o->v[0][i] = minimum_r;
        for (int q = 1; q < 7; q++) o->v[q][i] = 0.0;
    }
}
};

// count: N_MAX is to be counted from the radii (the step's sort has just left it)
hipError_t launch_potential(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub,
                            const Scratch &sc, hipStream_t st, bool count)
{
    const int64_t ntiles = n_ub > 0 ? (n_ub + CTILE - 1) / CTILE : 1;
    if (ntiles + 1 > sc.max_tiles) return hipErrorInvalidValue;
    // a test hook widens the classification's error bound, which sends the chains through
    // the repair
    PotArgs p;
    p.m = f.m; p.r = f.r; p.phi = f.phi; p.s = s;
    p.nstar = (double)P.n_star;
    p.xc = sc.chain_x;
    p.scal = sc.chain_scal;
    p.flag = sc.chain_fbad;
    p.nodes = sc.nodes;
    p.counted = count;
    p.a = esa_args(sc, P.chain_k_drop, 0);
    p.b = esa_args(sc, P.chain_k_drop, 1);
    p.a.sign = 1.0;
    p.b.sign = -1.0;
    p.c = p.a;                                       // A's tile sums and list are free when C needs its own
    p.c.raw_n = sc.esa_n + 3;
    p.a.s_n = sc.esa_n + 4;                          // walked at the same time as B's, for its last value alone
    p.a.s_idx = nullptr;
    const dim3 gt((unsigned)ntiles), bt(CT);
    const int self_prefix = ntiles <= SELF_PREFIX_MAX;
    if (count) {
        kl<pot_init_kernel>(dim3(1), dim3(1), 0, st, s);
        if (n_ub > 0) kl<pot_count_kernel>(dim3((unsigned)((n_ub + 255) / 256)), dim3(256), 0, st, (const double *)f.r, s);
    }
    kl<pot_sums_kernel>(gt, bt, 0, st, p);
    if (!self_prefix) {
        kl<esa_tile_scan_kernel>(dim3(1), dim3(WALK_T), 0, st, p.a, ntiles);
        kl<esa_tile_scan_kernel>(dim3(1), dim3(WALK_T), 0, st, p.b, ntiles);
    }
    kl<pot_classify_ab_kernel>(dim3((unsigned)(2 * ntiles)), bt, 0, st, p, P, self_prefix);
    kl<pot_walk_ab_kernel>(dim3(1), dim3(2 * CT), 0, st, p, P);
    kl<pot_rebuild_b_kernel>(gt, bt, 0, st, p);
    if (!self_prefix) kl<esa_tile_scan_kernel>(dim3(1), dim3(WALK_T), 0, st, p.c, ntiles);
    kl<pot_classify_c_kernel>(gt, bt, 0, st, p, self_prefix);
    kl<pot_walk_c_kernel>(dim3(1), bt, 0, st, p);
    kl<pot_rebuild_c_kernel>(gt, bt, 0, st, p, P);
    kl<pot_finish_kernel>(dim3(1), dim3(WALK_T), 0, st, p, P);
    return hipGetLastError();
}

hipError_t launch_potential_at(const DevFields &f, DevScalars *s, const KParams &P, const double *x,
                               double *out, int64_t count, hipStream_t st)
{
    (void)P;
    if (count <= 0) return hipSuccess;
    kl<pot_at_kernel>(dim3((unsigned)((count + 255) / 256)), dim3(256), 0, st, f.r, f.phi, s, x,
                       out, count);
    return hipGetLastError();
}

size_t report_work_bytes(const Scratch &sc) { return (size_t)REPORT_CHAINS * report_words(sc.max_tiles) * 8; }

// comp_mass_percent: pc (device, count <= MPC_MAX, ascending), results into out; work: the
// report workspace
hipError_t launch_mass_percent(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, const Scratch &sc,
                               const double *pc, int count, int bh_include, double itm, double minimum_r,
                               void *out, void *work, hipStream_t st)
{
    if (count < 0 || count > MPC_MAX) return hipErrorInvalidValue;
    int64_t ntiles = (n_ub + CTILE - 1) / CTILE + 1;
    if (ntiles > sc.max_tiles) return hipErrorInvalidValue;
    const int64_t xs = n_ub + 4, words = report_words(sc.max_tiles);
    const EsaArgs e = report_chain0(sc, P.chain_k_drop, work, xs);
    const double mprev0 = bh_include ? P.cenma_m * P.madhoc : 0.0;   // cmc_utils.c:878
    kl<mpc_prep_kernel>(dim3((unsigned)((n_ub + 256) / 256)), dim3(256), 0, st, f, (const DevScalars *)s, (double)P.n_star,
                       P.madhoc, mprev0, e, words, xs, (MassPcOut *)out);
    if (hipError_t err = run_chains(e, words, xs, 5, n_ub, st)) return err;
    kl<mpc_finish_kernel>(dim3(1), dim3(MPC_MAX), 0, st, (const double *)f.r, (const DevScalars *)s, (const double *)e.g, xs,
                       pc, count, bh_include, mprev0, itm, minimum_r, (MassPcOut *)out);
    return hipGetLastError();
}

size_t mass_percent_out_bytes() { return sizeof(MassPcOut); }

// ---------------------------------------------------------------- central_calculate
// cmc_utils.c:1239-1345 (J = 6) and clusdyn_calculate cmc_utils.c:1614-1624.  The
// half-mass index nave comes from the enclosed-mass chain of comp_mass_percent
// (star_m[k] / N_STAR, from 0); the six density-weighted sums over i = 1..nave are
// sequential recurrences solved by the exact chain emulation.  Each sum's terms are
// first scaled by a power of two that brings nave * max(term) to at most 1, so no
// partial sum can overflow; binary rounding is invariant under such a scaling, so the
// scaled chain rounds exactly as the unscaled one.
constexpr int CEN_TERMS = 6;     // rhoj, rhoj^2, rhoj v^2, rhoj r, (rhoj r)^2, rhoj m madhoc
enum { CEN_OK = 0, CEN_E_STATE = 1, CEN_E_RANGE = 2 };

struct CentralOut {
    int64_t nave;
    int32_t error, negative;     // negative: a mass is below zero (or NaN); 0 between calls
    double rh, rhojsum, rhoj2sum, rho, v_rms, rc, rc_nb, m_ave, n, rc_spitzer, N_core, N_core_nb, Trc;
    double S[CEN_TERMS];
    unsigned long long mx[CEN_TERMS];     // bit patterns of the terms' maxima (non-negative doubles)
    double scale[CEN_TERMS], unscale[CEN_TERMS];
};

// rhoj of cmc_utils.c:1263-1274 for star i: the 5 masses between jmin and jmax = jmin + 6
// over the shell volume between r[jmin] and r[jmax]
__device__ __forceinline__ double cen_rhoj(const double *__restrict__ r, const double *__restrict__ m,
                                           double madhoc, int64_t i)
{
    const double PI = 3.14159265358979323;                  // include/cmc/cmc.h:62
    const int64_t jmin = i - 3 > 1 ? i - 3 : 1, jmax = jmin + 6;
    double mrho = 0.0;
#pragma unroll
    for (int q = 1; q <= 5; q++) mrho += m[jmin + q] * madhoc;
    const double a = r[jmax], b = r[jmin];
    const double Vrj = 4.0 / 3.0 * PI * (a * a * a - b * b * b);
    return mrho / Vrj;
}

__device__ __forceinline__ void cen_terms(const DevFields &f, double madhoc, int64_t i, double (&v)[CEN_TERMS])
{
    const double rj = cen_rhoj(f.r, f.m, madhoc, i), r = f.r[i], vr = f.vr[i], vt = f.vt[i], q = rj * r;
    v[0] = rj;
    v[1] = rj * rj;
    v[2] = rj * (vr * vr + vt * vt);
    v[3] = q;
    v[4] = q * q;
    v[5] = rj * f.m[i] * madhoc;
}

// The enclosed-mass chain's increments star_m[k] / N_STAR from 0, the results and the
// start values cleared.
struct cen_begin_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ m, const DevScalars *s, double nstar,
                                  CentralOut *o, EsaArgs e, int64_t words)
{
    const int64_t j = (int64_t)kg_.bid * blockDim.x + threadIdx.x;
    const int64_t n = s->n_max;
    if (j == 0) {
        o->nave = 0;
        o->error = CEN_OK;
        *const_cast<int64_t *>(e.Lp) = n;
    }
    if (j < CEN_TERMS) {
        o->mx[j] = 0ull;
        o->S[j] = 0.0;
        o->scale[j] = o->unscale[j] = 1.0;
        const_cast<double *>(e.v0p)[j * words] = 0.0;
    }
    if (j < n) {
        const double mj = m[j + 1];
        const_cast<double *>(e.x)[j] = mj / nstar;
        if (!(mj >= 0.0)) o->negative = 1;
    }
}
};

// Smallest k in [lo, hi) for which pred (true, then false) fails, or hi, by a whole wave: 64
// probes split the range into 65.
template <class Pred>
__device__ __forceinline__ int64_t wave_first_false(int64_t lo, int64_t hi, Pred pred)
{
    const int lane = threadIdx.x & 63;
    while (lo < hi) {
        const int64_t step = (hi - lo) / 65 + 1, p = lo + (lane + 1) * step - 1;       // lo + 65 step > hi
        const int c = (int)__popcll(__ballot(p < hi && pred(p)));
        const int64_t top = lo + (c + 1) * step - 1;
        lo += c * step;
        hi = top < hi ? top : hi;
    }
    return lo;
}

// nave and rh from the chain g[k-1] = m after star k (cmc_utils.c:1247-1257, 1620-1623), by
// every block for itself: nave is the sums' length; then the terms' maxima.
struct cen_max_kernel {
    static constexpr int LB = 256, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const DevFields f, const DevScalars *s, const double *__restrict__ g,
                                  int64_t n_star, double madhoc, CentralOut *o, EsaArgs e, int64_t words)
{
    __shared__ unsigned long long red[CEN_TERMS][256 / 64];
    __shared__ int64_t found;
    const int64_t n = s->n_max;
    const double thr = 0.5 * s->Mtotal;
    if (threadIdx.x < 64) {
        // smallest k with !(g[k-1] < thr); g does not decrease, unless a mass is negative
        int64_t k = 1;
        if (!o->negative) {
            k = wave_first_false(1, n + 1, [&](int64_t q) { return g[q - 1] < thr; });
        } else {
            for (; k <= n; k += 64) {
                const uint64_t past = __ballot(k + threadIdx.x <= n && !(g[k + threadIdx.x - 1] < thr));
                if (past) {
                    k += __ffsll((unsigned long long)past) - 1;
                    break;
                }
            }
            if (k > n) k = n + 1;
        }
        if (threadIdx.x == 0) found = k;
    }
    __syncthreads();
    const int64_t k = found;
    const int64_t jmax_last = (k + 1 - 3 > 1 ? k + 1 - 3 : 1) + 6;
    const bool bad = k > n || n_star <= 12 || k + 1 >= n_star - 6 || jmax_last > n + 1;
    const int64_t nave = bad ? 0 : k + 1;
    if (kg_.bid == 0 && threadIdx.x < CEN_TERMS) {
        const_cast<int64_t *>(e.Lp)[threadIdx.x * words] = bad ? 1 : nave;    // bad: the sums run over one zero term
        if (threadIdx.x == 0) {
            o->nave = nave;
            if (bad) o->error = CEN_E_STATE;
            else o->rh = f.r[nave];
        }
    }
    unsigned long long mx[CEN_TERMS] = {0, 0, 0, 0, 0, 0};
    for (int64_t j = (int64_t)kg_.bid * blockDim.x + threadIdx.x; j < nave; j += (int64_t)kg_.nb * blockDim.x) {
        double v[CEN_TERMS];
        cen_terms(f, madhoc, j + 1, v);
        for (int t = 0; t < CEN_TERMS; t++) {
            const unsigned long long b = (unsigned long long)__double_as_longlong(v[t]);
            mx[t] = b > mx[t] ? b : mx[t];      // a negative or NaN term has the largest patterns
        }
    }
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int t = 0; t < CEN_TERMS; t++) {
        unsigned long long v = mx[t];
        for (int off = 32; off > 0; off >>= 1) {
            const unsigned long long u = __shfl_down(v, off, 64);
            v = u > v ? u : v;
        }
        if (lane == 0) red[t][w] = v;
    }
    __syncthreads();
    if (threadIdx.x < CEN_TERMS) {
        unsigned long long v = 0;
        for (int q = 0; q < 256 / 64; q++) v = red[threadIdx.x][q] > v ? red[threadIdx.x][q] : v;
        if (v) atomicMax(&o->mx[threadIdx.x], v);
    }
}
};

// The scales (by every block for itself; block 0 keeps them) and the scaled terms.
struct cen_prep_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const DevFields f, double madhoc, CentralOut *o, EsaArgs e, int64_t xs)
{
    __shared__ double scale[CEN_TERMS];
    __shared__ int range;
    const int t = threadIdx.x;
    const int64_t j = (int64_t)kg_.bid * blockDim.x + t, nave = o->nave;
    if (t == 0) range = 0;
    __syncthreads();
    if (t < CEN_TERMS) {
        const unsigned long long mx = o->mx[t];
        double up = 1.0, down = 1.0;
        if (mx >= 0x7ff0000000000000ull) {         // infinite, NaN or negative
            range = 1;
        } else {
            const double bound = (double)nave * __longlong_as_double((long long)mx);
            if (bound > 0.0) {
                int x;
                frexp(bound, &x);                  // bound <= 2^x
                down = ldexp(1.0, -x);
                up = ldexp(1.0, x);
            }
        }
        scale[t] = down;
        if (kg_.bid == 0) {
            o->scale[t] = down;
            o->unscale[t] = up;
        }
    }
    __syncthreads();
    if (range && kg_.bid == 0 && t == 0) o->error = CEN_E_RANGE;
    double *x = const_cast<double *>(e.x);
    if (nave == 0 || range) {                      // one zero term, or sums that are not used
        if (j < (nave > 0 ? nave : 1))
            for (int q = 0; q < CEN_TERMS; q++) x[q * xs + j] = 0.0;
        return;
    }
    if (j >= nave) return;
    double v[CEN_TERMS];
    cen_terms(f, madhoc, j + 1, v);
    for (int q = 0; q < CEN_TERMS; q++) {
        const double w = v[q] * scale[q];
        if (w != 0.0 && w < 2.2250738585072014e-308) o->error = CEN_E_RANGE;   // scaled into subnormals
        x[q * xs + j] = w;
    }
}
};

// the averages and derived quantities, cmc_utils.c:1323-1345
struct cen_final_kernel {
    static constexpr int LB = 64, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ g, int64_t xs, CentralOut *o)
{
    if (threadIdx.x == 0) o->negative = 0;
    if (o->error) return;
    if (threadIdx.x < CEN_TERMS) o->S[threadIdx.x] = g[threadIdx.x * xs + o->nave - 1] * o->unscale[threadIdx.x];
    __syncthreads();
    if (threadIdx.x != 0) return;
    const double PI = 3.14159265358979323;
    const double rhojsum = o->S[0], rhoj2sum = o->S[1];
    double rho = o->S[1], v_rms = o->S[2], rc = o->S[3], rc_nb = o->S[4], m_ave = o->S[5];
    rho /= rhojsum;
    rho *= 4.0 / 5.0;
    rho *= 2.0;
    v_rms /= rhojsum;
    v_rms = sqrt(v_rms);
    rc /= rhojsum;
    rc_nb = sqrt(rc_nb / rhoj2sum);
    m_ave /= rhojsum;
    const double n = rho / m_ave;
    o->rc_spitzer = sqrt(3.0 * (v_rms * v_rms) / (4.0 * PI * rho));
    o->N_core = 4.0 / 3.0 * PI * (rc * rc * rc) * (n / 2.0);
    o->N_core_nb = 4.0 / 3.0 * PI * (rc_nb * rc_nb * rc_nb) * (n / 2.0);
    o->Trc = 0.065 * (v_rms * v_rms * v_rms) / (rho * m_ave);
    o->rhojsum = rhojsum;
    o->rhoj2sum = rhoj2sum;
    o->rho = rho;
    o->v_rms = v_rms;
    o->rc = rc;
    o->rc_nb = rc_nb;
    o->m_ave = m_ave;
    o->n = n;
}
};

hipError_t launch_central(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, const Scratch &sc,
                          void *out, void *work, hipStream_t st)
{
    int64_t ntiles = (n_ub + CTILE - 1) / CTILE + 1;
    if (ntiles > sc.max_tiles) return hipErrorInvalidValue;
    const int64_t xs = n_ub + 4, words = report_words(sc.max_tiles);
    const EsaArgs e = report_chain0(sc, P.chain_k_drop, work, xs);
    CentralOut *o = (CentralOut *)out;
    const unsigned g1 = (unsigned)((n_ub + 256) / 256);
    kl<cen_begin_kernel>(dim3(g1), dim3(256), 0, st, (const double *)f.m, (const DevScalars *)s, (double)P.n_star, o, e, words);
    if (hipError_t err = run_chains(e, words, xs, 1, n_ub, st)) return err;
    const unsigned gmax = g1 < 1024u ? g1 : 1024u;
    kl<cen_max_kernel>(dim3(gmax), dim3(256), 0, st, f, (const DevScalars *)s, (const double *)e.g, (int64_t)P.n_star,
                       P.madhoc, o, e, words);
    kl<cen_prep_kernel>(dim3(g1), dim3(256), 0, st, f, P.madhoc, o, e, xs);
    if (hipError_t err = run_chains(e, words, xs, CEN_TERMS, n_ub, st)) return err;
    kl<cen_final_kernel>(dim3(1), dim3(64), 0, st, (const double *)e.g, xs, o);
    return hipGetLastError();
}

size_t central_out_bytes() { return sizeof(CentralOut); }
