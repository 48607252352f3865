// a1: qsorts_new -> sample_sort at one rank (src/cmc/cmc_sort.c:375-629): order the
// stars by r ascending (compare_type, :245-250), ties by id (the reference's libc
// qsort leaves them unordered), then by slot; drop the r == SF_INFINITY tail
// (remove_stripped_stars, :343-354), then refresh r and m (post_sort_comm,
// src/cmc/cmc_utils.c:2259-2288).
//
// Device algorithm: a distribution sort in two moves of each star's payload.
//   count    every star's bucket among B buckets of about SB_AVG stars and a bucket
//            histogram per tile;
//   scan     the tiles' offsets inside every bucket (only beyond SB_SMALL_N stars; below,
//            every scatter block sums the few histogram rows itself);
//   scatter  each star's fields packed into one 64- or 128-byte record at the next free
//            place of its bucket (order inside a bucket is free: the buckets are put into
//            the total order (r, id, slot) next, so the result does not depend on it);
//   sort     one block per bucket orders its records in LDS and writes every field
//            coalesced.
// In the step the bucket comes from the index of the new radius among the old ones, which
// the orbit phase found with the potential there: a step moves stars along their orbits
// and changes the density little, so equal cuts of the old order keep nearly equal counts.
// Where they would not (a cluster far from equilibrium: of a thin shell half the stars go
// inside every old radius), or the old radii do not ascend, the orbit phase has sampled the
// new radii, and the step bisects boundaries as the general entry point does, which orders
// radii it knows nothing about.  Counts decide only the speed: a bucket beyond the LDS capacity is
// split further by its block, in time proportional to its stars.
//
// Bound: HBM.  The payload (64 B a star) is read and written twice, 256 B a star, plus 4 B
// of node indices; the bucket pass reads the records a second time, in output order, mostly
// from the caches below the L2.  It replaced an LSD radix sort of (key, slot) words, which
// packed the records, moved the words through four histogram-scan-scatter passes and gathered
// the records at the end (16 launches, now 3 or 4).  The step's sort, before -> now: N = 1e4
// 0.099 -> 0.028 ms, 1e5 0.106 -> 0.034, 1e6 0.164 -> 0.092, 4e6 0.399 -> 0.282, 1.8e7
// 1.82 -> 1.28.  At 4e6 the scatter takes 112 us for 532 MB measured at the L2 (4.7 TB/s, the
// rate of a copy), the bucket pass 142 us for 889 MB (643 read, 245 written: 6.3 TB/s with
// what the caches serve, 3.6 of the 512 MB it cannot do without).
#include "kernels.hpp"

namespace {
constexpr int SB_MAX_FIELDS = 20;
// The payload without id: field f goes from src[f] to dst[f].
struct GatherList {
    int nf;
    const uint64_t *src[SB_MAX_FIELDS];
    uint64_t *dst[SB_MAX_FIELDS];
};

// Orders LDS traffic of one wave (its DS operations execute in order; this keeps the
// compiler from moving them).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Block-wide exclusive scan of one count per thread (lds: blockDim / 64 words, free on
// return); *total receives the sum.
__device__ __forceinline__ uint32_t block_excl(uint32_t v, uint32_t *lds, uint32_t *total)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(x, d, 64);
        if (lane >= d) x += y;
    }
    if (lane == 63) lds[w] = x;
    __syncthreads();
    uint32_t off = 0, tot = 0;
    for (int q = 0; q < nw; q++) {
        const uint32_t c = lds[q];
        if (q < w) off += c;
        tot += c;
    }
    __syncthreads();
    *total = tot;
    return off + x - v;
}

// Keys lo..hi cut into `bins` equal parts: a monotone map (the factor is rounded down, so
// every key stays below `bins`).
struct Binning {
    uint64_t lo, mult;
    int shift;
    __device__ __forceinline__ Binning(uint64_t lo_, uint64_t hi, int bins) : lo(lo_)
    {
        const uint64_t range = hi > lo ? hi - lo : 0;
        shift = range >> 32 ? 32 - __clzll((long long)range) : 0;
        mult = (uint64_t)((double)bins * 4294967296.0 / ((double)(range >> shift) + 1.0) * (1.0 - 0x1p-40));
    }
    __device__ __forceinline__ uint32_t operator()(uint64_t key) const { return (uint32_t)((((key - lo) >> shift) * mult) >> 32); }
};

// stars per tile when n stars are cut into nt tiles
__device__ __forceinline__ int64_t tile_chunk(int64_t n, int64_t nt) { return (n + nt - 1) / nt; }

// Bucket boundaries from a sample (the general entry point): S keys at even strides,
// ordered in LDS by a counting sort over sub-ranges and ranks inside them, or by a bitonic
// sort where a sub-range holds more than SMP_RANK of them (tied or clumped radii: the ranks
// among 8192 keys of one sub-range took 3.5 s); boundary b is the sample at rank b S / B.
constexpr int SMP_T = 1024, SMP_BINS = 4096, SMP_RANK = 64;
struct sb_sample_kernel {
    static constexpr int LB = SMP_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ keysrc, const DevScalars *s, int B,
                                               uint64_t *__restrict__ split, int32_t *__restrict__ moved)
{
    __shared__ uint64_t key[SMP_MAX];
    __shared__ uint32_t bin[SMP_BINS + 1];
    __shared__ uint64_t red[2][SMP_T / 64];
    __shared__ uint32_t scan[SMP_T / 64];
    __shared__ int clumped;
    const int t = threadIdx.x;
    const int64_t n = s->n_max_new;
    const int S = n < SMP_MAX ? (int)n : SMP_MAX;
    for (int q = t; q <= SMP_BINS; q += SMP_T) bin[q] = 0;
    if (t == 0) {
        clumped = 0;
        *moved = 0;
    }
    uint64_t k[SMP_MAX / SMP_T];
    uint64_t lo = ~0ull, hi = 0ull;
#pragma unroll
    for (int u = 0; u < SMP_MAX / SMP_T; u++) {
        const int q = u * SMP_T + t;
        k[u] = ~0ull;
        if (q < S) {
            k[u] = sortable(keysrc[1 + (int64_t)q * n / S]);
            if (k[u] > KEY_INF) k[u] = KEY_INF;               // the tail: one value above every live key
            lo = k[u] < lo ? k[u] : lo;
            hi = k[u] > hi ? k[u] : hi;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        const uint64_t a = __shfl_xor(lo, o, 64), b = __shfl_xor(hi, o, 64);
        lo = a < lo ? a : lo;
        hi = b > hi ? b : hi;
    }
    if ((t & 63) == 0) { red[0][t >> 6] = lo; red[1][t >> 6] = hi; }
    __syncthreads();
    for (int q = 0; q < SMP_T / 64; q++) {
        lo = red[0][q] < lo ? red[0][q] : lo;
        hi = red[1][q] > hi ? red[1][q] : hi;
    }
    const Binning bn_of(lo, hi, SMP_BINS);
    auto bin_of = [&](uint64_t x) { return bn_of(x); };
    uint32_t at[SMP_MAX / SMP_T];
#pragma unroll
    for (int u = 0; u < SMP_MAX / SMP_T; u++)
        if (u * SMP_T + t < S) at[u] = atomicAdd(&bin[bin_of(k[u])], 1u);
    __syncthreads();
    constexpr int PER = SMP_BINS / SMP_T;
    uint32_t c[PER], sum = 0, tot;
#pragma unroll
    for (int q = 0; q < PER; q++) {
        c[q] = bin[t * PER + q];
        sum += c[q];
        if (c[q] > SMP_RANK) clumped = 1;
    }
    uint32_t run = block_excl(sum, scan, &tot);
#pragma unroll
    for (int q = 0; q < PER; q++) { bin[t * PER + q] = run; run += c[q]; }
    if (t == 0) bin[SMP_BINS] = (uint32_t)S;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < SMP_MAX / SMP_T; u++)
        if (u * SMP_T + t < S) key[bin[bin_of(k[u])] + at[u]] = k[u];
    __syncthreads();
    if (clumped) {
        sample_sort(key, S);
        for (int b = t; b < B; b += SMP_T) split[b] = b > 0 ? key[(int64_t)b * S / B] : 0ull;
        return;
    }
    // boundary b: the sample of rank b S / B, found among its bin's keys
    for (int b = t; b < B; b += SMP_T) {
        uint64_t v = 0;
        if (b > 0 && S > 0) {
            const uint32_t rank = (uint32_t)((int64_t)b * S / B);
            const uint32_t bn = bin_of(key[rank]), e0 = bin[bn], e1 = bin[bn + 1];
            v = key[rank];
            for (uint32_t p = e0; p < e1; p++) {
                uint32_t less = 0;
                for (uint32_t q = e0; q < e1; q++) less += key[q] < key[p] || (key[q] == key[p] && q < p);
                if (e0 + less == rank) { v = key[p]; break; }
            }
        }
        split[b] = v;
    }
}
};

// Tile histograms over the buckets (row `tile` of mat), the step's form: buckets from the node
// indices, or, where these would be uneven, from the radii as in sb_count_kernel (the
// boundaries from memory: LDS for them would halve the blocks of the usual case).
template <int BM>
struct sb_count_step_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const int32_t *__restrict__ knew, DevScalars *s,
                                               const int32_t *__restrict__ uneven, int B, uint32_t *__restrict__ mat,
                                               const double *__restrict__ keysrc, const uint64_t *__restrict__ split,
                                               uint16_t *__restrict__ bkt)
{
    __shared__ uint32_t hist[BM];
    const int t = threadIdx.x;
    const int64_t n = s->n_max_new;
    if (kg_.bid == 0 && t == 0) s->sort_in = n;
    const StepBucket bucket(n, B);
    for (int b = t; b < B; b += 1024) hist[b] = 0;
    const int64_t chunk = tile_chunk(n, kg_.nb);
    const int64_t i0 = (int64_t)kg_.bid * chunk, i1 = i0 + chunk < n ? i0 + chunk : n;
    __syncthreads();
    if (*uneven) {
        for (int64_t i = i0 + t; i < i1; i += 1024) {
            const double x = keysrc[i + 1];
            const uint64_t k = sortable(x);
            uint32_t b = SB_TAIL;
            if (x < CMCG_SF_INFINITY) {                   // as the indices have it: not a NaN
                b = 0;
                for (int hi = B - 1; (int)b < hi;) {
                    const int m = ((int)b + hi + 1) >> 1;
                    if (split[m] <= k) b = m;
                    else hi = m - 1;
                }
                atomicAdd(&hist[b], 1u);
            }
            bkt[i] = (uint16_t)b;
        }
    } else {
        for (int64_t c = i0; c < i1; c += 4 * 1024) {
            int32_t k[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {                 // independent loads in flight
                const int64_t i = c + u * 1024 + t;
                k[u] = i < i1 ? knew[i + 1] : -1;
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if (k[u] >= 0) atomicAdd(&hist[bucket(k[u])], 1u);
        }
    }
    __syncthreads();
    for (int b = t; b < B; b += 1024) mat[(int64_t)kg_.bid * B + b] = hist[b];
}
};

// The same from the radii, and every star's bucket: the number of boundaries
// split[1..B-1] at or below its key; *moved where a live star is not at its place among its
// neighbours.
template <int BM>
struct sb_count_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ keysrc, DevScalars *s,
                                               const uint64_t *__restrict__ split, int B, uint16_t *__restrict__ bkt,
                                               uint32_t *__restrict__ mat, const int64_t *__restrict__ id, int32_t *moved)
{
    __shared__ uint64_t spl[BM];
    __shared__ uint32_t hist[BM];
    const int t = threadIdx.x;
    const int64_t n = s->n_max_new;
    if (kg_.bid == 0 && t == 0) s->sort_in = n;
    for (int b = t; b < B; b += 1024) {
        spl[b] = split[b];
        hist[b] = 0;
    }
    int top = 1;
    while (top < B) top <<= 1;
    const int64_t chunk = tile_chunk(n, kg_.nb);
    const int64_t i0 = (int64_t)kg_.bid * chunk, i1 = i0 + chunk < n ? i0 + chunk : n;
    bool out = false;
    __syncthreads();
    for (int64_t c = i0; c < i1; c += 4 * 1024) {
        uint64_t k[4], before[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {                     // independent loads in flight
            const int64_t i = c + u * 1024 + t;
            k[u] = i < i1 ? sortable(keysrc[i + 1]) : ~0ull;
            before[u] = i < i1 && i > 0 ? sortable(keysrc[i]) : 0ull;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int64_t i = c + u * 1024 + t;
            if (k[u] < KEY_INF && (before[u] > k[u] || (before[u] == k[u] && id[i] > id[i + 1]))) out = true;
        }
        int at[4] = {0, 0, 0, 0};
        for (int st = top >> 1; st > 0; st >>= 1) {
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int m = at[u] + st;
                if (m < B && spl[m] <= k[u]) at[u] = m;
            }
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int64_t i = c + u * 1024 + t;
            if (i >= i1) continue;
            const bool live = k[u] < KEY_INF;
            bkt[i] = live ? (uint16_t)at[u] : SB_TAIL;
            if (live) atomicAdd(&hist[at[u]], 1u);
        }
    }
    if (out) *moved = 1;
    __syncthreads();
    for (int b = t; b < B; b += 1024) mat[(int64_t)kg_.bid * B + b] = hist[b];
}
};

// The tiles' exclusive offsets inside every bucket, in place, and the bucket totals.  A
// block takes 64 buckets; its 16 waves take consecutive groups of tiles, lane = bucket.
struct sb_scan_kernel {
    static constexpr int LB = 1024, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, uint32_t *__restrict__ mat, uint32_t *__restrict__ totals, int B,
                                               int nt)
{
    constexpr int PER = SB_MAX_TILES / 16;
    __shared__ uint32_t part[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int b = kg_.bid * 64 + lane;
    const int per = (nt + 15) / 16, t0 = w * per;
    uint32_t c[PER], sum = 0;
#pragma unroll
    for (int q = 0; q < PER; q++) {
        c[q] = q < per && t0 + q < nt && b < B ? mat[(int64_t)(t0 + q) * B + b] : 0u;
        sum += c[q];
    }
    part[w][lane] = sum;
    __syncthreads();
    uint32_t run = 0, tot = 0;
    for (int q = 0; q < 16; q++) {
        if (q < w) run += part[q][lane];
        tot += part[q][lane];
    }
#pragma unroll
    for (int q = 0; q < PER; q++)
        if (q < per && t0 + q < nt && b < B) {
            mat[(int64_t)(t0 + q) * B + b] = run;
            run += c[q];
        }
    if (w == 0 && b < B) totals[b] = tot;
}
};

// Records of W words: r, id, slot, then the first W - 3 payload fields.  A wave packs 64
// stars at a time through its own LDS patch (odd stride: no bank conflicts), so whole
// records leave in each store instruction; the next 64 stars' loads are in flight
// meanwhile.  knew: the step's form (bkt is read only where the indices would be uneven).
// scanned: mat holds the tiles' offsets and totals the bucket totals (sb_scan_kernel);
// otherwise both are formed here from the raw histogram rows.  Bound by HBM: 532 MB in
// 112 us at N = 4e6.
constexpr int SC_T = 512, SC_W = SC_T / 64;
template <int W, int BM>
struct sb_scatter_kernel {
    static constexpr int LB = SC_T, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const double *__restrict__ keysrc,
                                               const uint64_t *__restrict__ id, const DevScalars *s,
                                               const uint16_t *__restrict__ bkt, const int32_t *__restrict__ knew,
                                               const int32_t *__restrict__ uneven, const uint32_t *__restrict__ mat,
                                               const uint32_t *__restrict__ totals, uint32_t *__restrict__ first, int B,
                                               int scanned, uint64_t *__restrict__ aos, GatherList g,
                                               const int32_t *__restrict__ moved)
{
    constexpr int NF = W - 3, LD = W + 1, PC = W / 2;
    static_assert(SB_SMALL_BUCKETS <= SC_T, "one bucket per thread without the scan pass");
    __shared__ uint32_t next[BM];
    __shared__ uint64_t patch[SC_W][64 * LD];
    __shared__ uint32_t place[SC_W][64];
    __shared__ uint32_t lds[SC_W];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int64_t n = s->n_max_new;
    const int tile = kg_.bid, nt = kg_.nb;
    // the tile's first free place in every bucket; tile 0 also writes the buckets' first
    // places and the number of stars to first[0..B].  Every load is issued before the first
    // use (a thread's buckets one after another would cost a memory latency each).
    {
        constexpr int PER = (BM + SC_T - 1) / SC_T;
        const int per = (B + SC_T - 1) / SC_T;
        uint32_t tot[PER], off[PER], sum = 0, all;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int b = t * per + q;
            const bool in = q < per && b < B;
            tot[q] = in && scanned ? totals[b] : 0u;
            off[q] = in && scanned ? mat[(int64_t)tile * B + b] : 0u;
        }
        if (!scanned && t < B) {                           // B <= SC_T here: one bucket per thread
            uint32_t c[SB_SMALL_TILES];
#pragma unroll
            for (int r = 0; r < SB_SMALL_TILES; r++) c[r] = r < nt ? mat[(int64_t)r * B + t] : 0u;
#pragma unroll
            for (int r = 0; r < SB_SMALL_TILES; r++) {
                if (r < tile) off[0] += c[r];
                tot[0] += c[r];
            }
        }
#pragma unroll
        for (int q = 0; q < PER; q++) sum += tot[q];
        uint32_t base = block_excl(sum, lds, &all);
#pragma unroll
        for (int q = 0; q < PER; q++) {
            const int b = t * per + q;
            if (q < per && b < B) {
                next[b] = base + off[q];
                if (tile == 0) first[b] = base;
            }
            base += tot[q];
        }
        if (tile == 0 && t == 0) first[B] = all;
        __syncthreads();
    }
    if (moved && !*moved) return;                          // in order: the bucket pass copies the fields
    const int64_t chunk = tile_chunk(n, nt);
    const int64_t i0 = (int64_t)tile * chunk, i1 = i0 + chunk < n ? i0 + chunk : n;
    const StepBucket bucket(n, B);
    const bool by_index = knew && !*uneven;
    uint64_t v[NF], kr = 0, vid = 0;
    uint32_t bk = SB_TAIL;
    auto load = [&](int64_t i) {
        bk = SB_TAIL;
        if (i < i1) {
            bk = by_index ? bucket(knew[i + 1]) : bkt[i];
            kr = (uint64_t)__double_as_longlong(keysrc[i + 1]);
            vid = id[i + 1];
#pragma unroll
            for (int f = 0; f < NF; f++) v[f] = f < g.nf ? g.src[f][i + 1] : 0ull;
        }
    };
    uint64_t *mine = patch[w];
    load(i0 + w * 64 + lane);
    for (int64_t c = i0 + w * 64; c < i1; c += SC_T) {             // wave-uniform
        uint32_t p = ~0u;
        if (bk != SB_TAIL) {
            p = atomicAdd(&next[bk], 1u);
            mine[LD * lane] = kr;
            mine[LD * lane + 1] = vid;
            mine[LD * lane + 2] = (uint64_t)(c + lane + 1);
#pragma unroll
            for (int f = 0; f < NF; f++) mine[LD * lane + 3 + f] = v[f];
        }
        place[w][lane] = p;
        load(c + SC_T + lane);
        wave_sync();
#pragma unroll
        for (int u = 0; u < PC; u++) {
            const int task = u * 64 + lane, rec = task / PC, pc = task % PC;
            const uint32_t q = place[w][rec];
            if (q != ~0u)
                *(ulonglong2 *)(aos + (int64_t)W * q + 2 * pc) =
                    ulonglong2{mine[LD * rec + 2 * pc], mine[LD * rec + 2 * pc + 1]};
        }
        wave_sync();
    }
}
};

// ---------------------------------------------------------------- one bucket
// Records a, b of a bucket in the order (r, id, slot).
template <int W>
__device__ __forceinline__ bool rec_less(const uint64_t *__restrict__ rec, uint32_t a, uint32_t b)
{
    const uint64_t *x = rec + (int64_t)W * a, *y = rec + (int64_t)W * b;
    const uint64_t ka = sortable(__longlong_as_double((long long)x[0])), kb = sortable(__longlong_as_double((long long)y[0]));
    if (ka != kb) return ka < kb;
    const int64_t ia = (int64_t)x[1], ib = (int64_t)y[1];
    return ia < ib || (ia == ib && x[2] < y[2]);
}

// word w of record a as an unsigned key: the order (r, id, slot) word by word
template <int W>
__device__ __forceinline__ uint64_t rec_key(const uint64_t *__restrict__ rec, uint32_t a, int w)
{
    const uint64_t x = rec[(int64_t)W * a + w];
    return w == 0 ? sortable(__longlong_as_double((long long)x)) : w == 1 ? x ^ 0x8000000000000000ull : x;
}

// Some records of a bucket: those that a list names, or (no list) all of them.
struct Records {
    const uint32_t *list;
    __device__ __forceinline__ uint32_t operator()(uint32_t e) const { return list ? list[e] : e; }
};

constexpr int BS_T = 512, BS_BINS = 2048, BS_RANK = 48;
constexpr int SPLIT_BINS = 1024;        // parts of one split of a bucket beyond the LDS capacity

template <int W, int CAP>
struct BucketLds {
    static constexpr int PC = W / 2, SN = 256 * 8 / W;              // records staged at a time: 16 KB
    static constexpr int STAGE = SN * PC + SN * PC / 32;            // 16-byte pieces, one pad per 32
    static constexpr int BUF = 2 * STAGE > CAP ? 2 * STAGE : CAP;
    static_assert(CAP % BS_T == 0 && (CAP & (CAP - 1)) == 0, "LDS capacity");
    __align__(16) uint64_t buf[BUF];                                // keys, later the staged records
    uint16_t idx[CAP], fin[CAP];
    uint32_t bin[BS_BINS + 1], sub[SPLIT_BINS];
    uint32_t scan[BS_T / 64];
    uint64_t red[2][BS_T / 64];
    uint32_t worst;
};

// Bitonic sort in LDS of the first cnt entries (cnt <= CAP, a power of two), idx numbering
// the records of `of`; the rest of the next power of two is padded with entries above every record.
template <int W>
__device__ void bitonic(const uint64_t *__restrict__ rec, const Records &of, uint64_t *key, uint16_t *idx, int cnt)
{
    int P = 1, t = threadIdx.x;
    asm volatile("" : "+v"(t));
    while (P < cnt) P <<= 1;
    for (int q = cnt + t; q < P; q += BS_T) { key[q] = ~0ull; idx[q] = 0xffff; }
    __syncthreads();
    for (int kk = 2; kk <= P; kk <<= 1)
        for (int j = kk >> 1; j > 0; j >>= 1) {
            for (int q = t; q < P; q += BS_T) {
                const int x = q ^ j;
                if (x > q) {
                    const uint64_t ka = key[q], kb = key[x];
                    const uint16_t a = idx[q], b = idx[x];
                    const bool up = (q & kk) == 0;
                    const bool gt = kb < ka || (kb == ka && b != 0xffff && (a == 0xffff || rec_less<W>(rec, of(b), of(a))));
                    if (gt == up) { key[q] = kb; key[x] = ka; idx[q] = b; idx[x] = a; }
                }
            }
            __syncthreads();
        }
}

// values that every lane of the block holds, as the scalars they are
__device__ __forceinline__ uint32_t uniform(uint32_t x) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)x); }
__device__ __forceinline__ uint64_t uniform(uint64_t x) { return (uint64_t)uniform((uint32_t)(x >> 32)) << 32 | uniform((uint32_t)x); }

// sh.red's wave values folded: the least and the greatest key over the block
template <class Lds>
__device__ __forceinline__ void block_range(Lds &sh, uint64_t &lo, uint64_t &hi)
{
    for (int o = 32; o > 0; o >>= 1) {
        const uint64_t x = __shfl_xor(lo, o, 64), y = __shfl_xor(hi, o, 64);
        lo = x < lo ? x : lo;
        hi = y > hi ? y : hi;
    }
    if ((threadIdx.x & 63) == 0) { sh.red[0][threadIdx.x >> 6] = lo; sh.red[1][threadIdx.x >> 6] = hi; }
    __syncthreads();
    for (int q = 0; q < BS_T / 64; q++) {
        lo = sh.red[0][q] < lo ? sh.red[0][q] : lo;
        hi = sh.red[1][q] > hi ? sh.red[1][q] : hi;
    }
    lo = uniform(lo);
    hi = uniform(hi);
}

// The order of cnt <= CAP records of a bucket in LDS: sh.fin[rank] = e for record of(e).
// They agree in the words before w.  The keys are counted into BS_BINS equal parts of their
// range, placed part by part, and each takes its rank among the few keys of its part; a part
// of more than BS_RANK keys (many equal radii, a very uneven bucket) sends them through the
// bitonic sort instead.
template <int W, int CAP>
__device__ __forceinline__ void order_records(const uint64_t *__restrict__ rec, const Records &of, int cnt, int w,
                                              BucketLds<W, CAP> &sh)
{
    constexpr int ITEMS = CAP / BS_T;
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    uint64_t k[ITEMS], lo = ~0ull, hi = 0ull;
    uint32_t at[ITEMS];
#pragma unroll
    for (int u = 0; u < ITEMS; u++) {
        const int e = u * BS_T + t;
        k[u] = 0;
        if (e < cnt) {
            k[u] = rec_key<W>(rec, of(e), w);
            lo = k[u] < lo ? k[u] : lo;
            hi = k[u] > hi ? k[u] : hi;
        }
    }
    for (int q = t; q <= BS_BINS; q += BS_T) sh.bin[q] = 0;
    if (t == 0) sh.worst = 0;
    block_range(sh, lo, hi);
    const Binning bin_of(lo, hi, BS_BINS);
#pragma unroll
    for (int u = 0; u < ITEMS; u++)
        if (u * BS_T + t < cnt) at[u] = atomicAdd(&sh.bin[bin_of(k[u])], 1u);
    __syncthreads();
    constexpr int PER = BS_BINS / BS_T;
    uint32_t c[PER], sum = 0, mx = 0, dummy;
#pragma unroll
    for (int q = 0; q < PER; q++) {
        c[q] = sh.bin[t * PER + q];
        sum += c[q];
        mx = c[q] > mx ? c[q] : mx;
    }
    if (mx > BS_RANK) sh.worst = mx;                       // any value above BS_RANK will do
    uint32_t run = block_excl(sum, sh.scan, &dummy);
#pragma unroll
    for (int q = 0; q < PER; q++) { sh.bin[t * PER + q] = run; run += c[q]; }
    if (t == 0) sh.bin[BS_BINS] = (uint32_t)cnt;
    __syncthreads();
    const bool uneven = uniform(sh.worst) > BS_RANK;
#pragma unroll
    for (int u = 0; u < ITEMS; u++) {
        const int e = u * BS_T + t;
        if (e < cnt) {
            const uint32_t p = uneven ? (uint32_t)e : sh.bin[bin_of(k[u])] + at[u];
            sh.buf[p] = k[u];
            sh.idx[p] = (uint16_t)e;
            at[u] = p;
        }
    }
    __syncthreads();
    if (uneven) {
        bitonic<W>(rec, of, sh.buf, sh.idx, cnt);
        for (int q = t; q < cnt; q += BS_T) sh.fin[q] = sh.idx[q];
    } else {
#pragma unroll
        for (int u = 0; u < ITEMS; u++) {
            const int e = u * BS_T + t;
            if (e < cnt) {
                const uint32_t bn = bin_of(k[u]), e0 = sh.bin[bn], e1 = sh.bin[bn + 1];
                uint32_t rank = e0;
                for (uint32_t q = e0; q < e1; q++)
                    if (q != at[u])
                        rank += sh.buf[q] < k[u] || (sh.buf[q] == k[u] && rec_less<W>(rec, of(sh.idx[q]), of((uint32_t)e)));
                sh.fin[rank] = (uint16_t)e;
            }
        }
    }
    __syncthreads();
}

// A bucket beyond the LDS capacity is ordered by its block in time proportional to its
// records, whatever their radii: their numbers are split into SPLIT_BINS equal parts of their
// key range, in key order; runs of parts that fit are ordered in LDS, and a part that does
// not is split again, by its narrower range or, all its keys equal, by the next word (ids, then
// slots, which differ).
// A part that waits has its numbers in one of (ord, tmp) and a note at the same place of the
// other one: the part that waits after it (place and array), its length and its word.
// (Buckets grow beyond their 1024 records where the cluster is far from equilibrium, where
// radii are tied, and all of them from 8.4e6 stars on, when there are as many as there may be.)
struct Part {
    uint32_t start, len;
    int w, in;                                             // numbers: 0 in ord, 1 in tmp, 2 all records
};
// The numbers of part p to the other array, part by part; sh.sub[b] is the end of its part b.
template <int W, class Lds>
__device__ __forceinline__ void split_part(const uint64_t *__restrict__ rec, Part &p, uint32_t *ord, uint32_t *tmp, Lds &sh)
{
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    const Records of{p.in == 2 ? nullptr : (p.in ? tmp : ord) + p.start};
    uint64_t lo, hi;
    for (;; p.w++) {
        lo = ~0ull;
        hi = 0ull;
#pragma unroll 2
        for (uint32_t e = t; e < p.len; e += BS_T) {
            const uint64_t k = rec_key<W>(rec, of(e), p.w);
            lo = k < lo ? k : lo;
            hi = k > hi ? k : hi;
        }
        for (int q = t; q < SPLIT_BINS; q += BS_T) sh.sub[q] = 0;
        block_range(sh, lo, hi);
        if (lo < hi || p.w == 2) break;
        __syncthreads();
    }
    const Binning bin_of(lo, hi, SPLIT_BINS);
#pragma unroll 2
    for (uint32_t e = t; e < p.len; e += BS_T) atomicAdd(&sh.sub[bin_of(rec_key<W>(rec, of(e), p.w))], 1u);
    __syncthreads();
    constexpr int PER = SPLIT_BINS / BS_T;
    uint32_t c[PER], sum = 0, dummy;
#pragma unroll
    for (int q = 0; q < PER; q++) { c[q] = sh.sub[t * PER + q]; sum += c[q]; }
    uint32_t run = block_excl(sum, sh.scan, &dummy);
#pragma unroll
    for (int q = 0; q < PER; q++) { sh.sub[t * PER + q] = run; run += c[q]; }
    __syncthreads();
    p.in = p.in == 0 ? 1 : 0;
    uint32_t *to = (p.in ? tmp : ord) + p.start;
#pragma unroll 2
    for (uint32_t e = t; e < p.len; e += BS_T) {
        const uint32_t a = of(e);
        to[atomicAdd(&sh.sub[bin_of(rec_key<W>(rec, a, p.w))], 1u)] = a;
    }
    __syncthreads();
}

// The order of a bucket's cnt records: in sh.fin up to CAP of them, else in ord.
template <int W, int CAP>
__device__ __forceinline__ void order_bucket(const uint64_t *__restrict__ rec, uint32_t cnt, uint32_t *ord, uint32_t *tmp,
                                             BucketLds<W, CAP> &sh)
{
    constexpr uint64_t NONE = ~0ull, WHOLE = ~1ull;
    Part p{0, 0, 0, 2};
    uint64_t waiting = WHOLE;                              // 2 place + array
    uint32_t s = 0, e = 0;                                 // the run of p in hand
    int b = 0;
    const bool fits = cnt <= CAP;
    if (fits) {
        order_records<W, CAP>(rec, Records{nullptr}, cnt, 0, sh);
        return;
    }
    for (;;) {
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));                        // keeps what depends on it out of registers between runs
        // the next run: parts b .. b1 - 1 fit together
        s = e;
        if (s == p.len) {
            if (waiting == NONE) return;
            __syncthreads();
            if (waiting == WHOLE) {
                waiting = NONE;
                p.len = cnt;
            } else {
                p.in = (int)(waiting & 1);
                p.start = (uint32_t)(waiting >> 1);
                const uint32_t *note = (p.in ? ord : tmp) + p.start;
                waiting = uniform(note[0]) | (uint64_t)uniform(note[1]) << 32;
                p.len = uniform(note[2]);
                p.w = (int)uniform(note[3]);
                __syncthreads();                       // the split writes where the note is
            }
            split_part<W>(rec, p, ord, tmp, sh);
            s = 0;
            b = 0;
        }
        int b1 = b, top = SPLIT_BINS;
        while (b1 < top) {
            const int m = (b1 + top) >> 1;
            if (uniform(sh.sub[m]) - s <= CAP) b1 = m + 1;
            else top = m;
        }
        if (b1 == b) {                                 // part b alone is too long: it waits
            e = uniform(sh.sub[b]);
            if (t == 0) {
                uint32_t *note = (p.in ? ord : tmp) + p.start + s;
                note[0] = (uint32_t)waiting;
                note[1] = (uint32_t)(waiting >> 32);
                note[2] = e - s;
                note[3] = (uint32_t)p.w;
            }
            waiting = 2 * (uint64_t)(p.start + s) + p.in;
            b++;
            continue;
        }
        e = uniform(sh.sub[b1 - 1]);
        b = b1;
        if (e == s) continue;
        const int m = (int)(e - s);
        const Records of{(p.in ? tmp : ord) + p.start + s};
        // (with 2048 records in LDS four blocks share a compute unit, which leaves 64 registers:
        // the counting order's keys and places do not fit them inside this loop)
        if (CAP > 2048) {
            order_records<W, CAP>(rec, of, m, p.w, sh);
        } else {
            for (int q = t; q < m; q += BS_T) {
                sh.buf[q] = rec_key<W>(rec, of.list[q], p.w);
                sh.idx[q] = (uint16_t)q;
            }
            bitonic<W>(rec, of, sh.buf, sh.idx, m);
            for (int q = t; q < m; q += BS_T) sh.fin[q] = sh.idx[q];
            __syncthreads();
        }
        uint32_t v[CAP / BS_T];
#pragma unroll
        for (int u = 0; u < CAP / BS_T; u++)
            if (u * BS_T + t < m) v[u] = of(sh.fin[u * BS_T + t]);
        __syncthreads();                                   // the numbers may be in ord
#pragma unroll
        for (int u = 0; u < CAP / BS_T; u++)
            if (u * BS_T + t < m) ord[p.start + s + u * BS_T + t] = v[u];
        __syncthreads();
    }
}

// Block b orders bucket b and writes its stars' fields: the sorted records are read back in
// output order, W/2 lanes per record, and leave through LDS with one coalesced store per
// field.  (The general entry point's stars are often in order already; then the blocks only
// copy them: 0.65 -> 0.45 ms at N = 4e6, 0.22 -> 0.16 at 1e6.)  Bound by HBM (N = 4e6, 8 words:
// 142 us); holding the records in registers between the two reads, or 256 threads a block,
// changed nothing.
template <int W, int CAP>
struct sb_sort_kernel {
    static constexpr int LB = BS_T, MB = CAP <= 2048 ? 8 : 4;
    static __device__ __forceinline__ void run(KGrid kg_, DevScalars *s, const uint32_t *__restrict__ place,
                                               const uint64_t *__restrict__ aos, uint32_t *order, int64_t n_cap,
                                               double *__restrict__ r_out, uint64_t *__restrict__ id_out,
                                               uint32_t *__restrict__ perm, GatherList g,
                                               const double *__restrict__ keysrc, const uint64_t *__restrict__ id,
                                               const int32_t *__restrict__ moved)
{
    using Lds = BucketLds<W, CAP>;
    constexpr int NF = W - 3, PC = Lds::PC, SN = Lds::SN;
    __shared__ Lds sh;
    const int t = threadIdx.x, nb = kg_.nb, b = kg_.bid;
    const uint32_t first = place[b], mine = place[b + 1] - first;
    if (b == 0 && t == 0) {
        const uint32_t tot = place[nb];
        s->sort_n = tot;
        s->n_max = tot;
        s->n_max_new = tot;                                // no block of this launch reads them
        r_out[(int64_t)tot + 1] = CMCG_SF_INFINITY;        // the outer sentinel (potential_calculate sets it again)
    }
    if constexpr (W == 16) {
        if (moved && !*moved) {                            // in order: block b copies its share of the fields
            const int64_t live = place[nb], share = tile_chunk(live, nb), i0 = b * share;
            for (int64_t i = i0 + t; i < i0 + share && i < live; i += BS_T) {
                r_out[i + 1] = keysrc[i + 1];
                id_out[i + 1] = id[i + 1];
                perm[i] = (uint32_t)(i + 1);
#pragma unroll
                for (int f = 0; f < NF; f++)
                    if (f < g.nf) g.dst[f][i + 1] = g.src[f][i + 1];
            }
            return;
        }
    }
    if (!mine) return;
    const int64_t cnt = mine;
    const uint64_t *rec = aos + (int64_t)W * first;
    const uint32_t *ord = cnt > CAP ? order + first : nullptr;
    order_bucket<W, CAP>(rec, mine, order + first, order + n_cap + first, sh);
    ulonglong2 *stage = (ulonglong2 *)sh.buf;
    for (int64_t c0 = 0; c0 < cnt; c0 += SN) {
        const int live = (int)(cnt - c0 < SN ? cnt - c0 : SN);
#pragma unroll
        for (int u = 0; u < SN * PC / BS_T; u++) {
            const int task = u * BS_T + t, sl = task / PC, pc = task % PC;
            if (sl < live) {
                const uint32_t e = ord ? ord[c0 + sl] : sh.fin[c0 + sl];
                stage[task + task / 32] = *(const ulonglong2 *)(rec + (int64_t)W * e + 2 * pc);
            }
        }
        __syncthreads();
        if (t < live) {
            uint64_t w[W];
#pragma unroll
            for (int q = 0; q < PC; q++) {
                const int task = t * PC + q;
                const ulonglong2 x = stage[task + task / 32];
                w[2 * q] = x.x;
                w[2 * q + 1] = x.y;
            }
            const int64_t i = (int64_t)first + c0 + t;
            r_out[i + 1] = __longlong_as_double((long long)w[0]);
            id_out[i + 1] = w[1];
            perm[i] = (uint32_t)w[2];
#pragma unroll
            for (int f = 0; f < NF; f++)
                if (f < g.nf) g.dst[f][i + 1] = w[3 + f];
        }
        __syncthreads();
    }
}
};

// The payload fields beyond a record's, through the permutation.
struct sb_rest_kernel {
    static constexpr int LB = 256, MB = 0;
    static __device__ __forceinline__ void run(KGrid kg_, const DevScalars *s, const uint32_t *__restrict__ perm, int f0,
                                               GatherList g)
{
    const int64_t i = (int64_t)kg_.bid * 256 + threadIdx.x;
    if (i >= s->sort_n) return;
    const uint32_t src = perm[i];
    for (int f = f0; f < g.nf; f++) g.dst[f][i + 1] = g.src[f][src];
}
};

template <int W, int BM, int CAP>
hipError_t sort_launch(const double *key_src, double *r_dst, const uint64_t *id_src, uint64_t *id_dst, const GatherList &g,
                       DevScalars *s, const Scratch &sc, const SortShape &sh, int64_t n_ub, const int32_t *knew,
                       hipStream_t st)
{
    if (knew) {
        kl<sb_count_step_kernel<BM>>(dim3((unsigned)sh.tiles), dim3(1024), 0, st, knew, s, (const int32_t *)sc.sort_uneven,
                                     sh.buckets, sc.sort_mat, key_src, (const uint64_t *)sc.sort_split, sc.sort_bkt);
    } else {
        kl<sb_sample_kernel>(dim3(1), dim3(SMP_T), 0, st, key_src, (const DevScalars *)s, sh.buckets, sc.sort_split,
                             sc.sort_moved);
        kl<sb_count_kernel<BM>>(dim3((unsigned)sh.tiles), dim3(1024), 0, st, key_src, s, (const uint64_t *)sc.sort_split,
                                sh.buckets, sc.sort_bkt, sc.sort_mat, (const int64_t *)id_src, sc.sort_moved);
    }
    const int32_t *moved = knew || W < 16 ? nullptr : sc.sort_moved;      // wide payloads alone are copied
    const int scanned = !sh.small;
    if (scanned)
        kl<sb_scan_kernel>(dim3((unsigned)((sh.buckets + 63) / 64)), dim3(1024), 0, st, sc.sort_mat, sc.sort_tot,
                           sh.buckets, sh.tiles);
    kl<sb_scatter_kernel<W, BM>>(dim3((unsigned)sh.tiles), dim3(SC_T), 0, st, key_src, id_src, (const DevScalars *)s,
                                 (const uint16_t *)sc.sort_bkt, knew, (const int32_t *)sc.sort_uneven,
                                 (const uint32_t *)sc.sort_mat, (const uint32_t *)sc.sort_tot, sc.sort_first, sh.buckets,
                                 scanned, sc.sort_aos, g, moved);
    kl<sb_sort_kernel<W, CAP>>(dim3((unsigned)sh.buckets), dim3(BS_T), 0, st, s, (const uint32_t *)sc.sort_first,
                               (const uint64_t *)sc.sort_aos, sc.sort_order, sc.sort_aos_cap, r_dst, id_dst, sc.vals_a, g,
                               key_src, id_src, moved);
    if (g.nf > W - 3 && n_ub > 0)
        kl<sb_rest_kernel>(dim3((unsigned)((n_ub + 255) / 256)), dim3(256), 0, st, (const DevScalars *)s,
                           (const uint32_t *)sc.vals_a, W - 3, g);
    return hipGetLastError();
}
} // namespace

// Sort slots 1..n_max_new by (key field, id).  src/dst are parallel lists of payload
// fields, id the last of them; key_src is the field holding the radii to sort by; r_dst
// receives them sorted.  knew: the radii's indices among the old nodes that the orbit
// phase left (the step's sort), or null.
hipError_t launch_sort_fields(const double *key_src, double *r_dst, int nf, const uint64_t *const *src,
                              uint64_t *const *dst, DevScalars *s, const Scratch &sc, int64_t n_ub,
                              const int32_t *knew, hipStream_t st)
{
    if (nf < 1 || nf - 1 > SB_MAX_FIELDS || n_ub > sc.sort_aos_cap) return hipErrorInvalidValue;
    GatherList g{};
    g.nf = nf - 1;
    for (int f = 0; f < g.nf; f++) { g.src[f] = src[f]; g.dst[f] = dst[f]; }
    const SortShape sh = sort_shape(n_ub);
    if ((size_t)sh.tiles * sh.buckets > sc.sort_mat_cap) return hipErrorInvalidValue;
    const uint64_t *id_src = src[nf - 1];
    uint64_t *id_dst = dst[nf - 1];
    // Records: 8 words hold r, id, slot and five fields (the step's sort); a wider payload
    // takes 16 words, and its buckets, cut from a sample, get twice the LDS capacity.  So do
    // the step's where SB_MAX_BUCKETS of SB_AVG stars are not enough: its sort at 1.8e7 stars
    // 1.70 ms with 2048 records in LDS, 1.28 with 4096; 3.90 and 3.44 at 3.6e7, 8.6 and 7.9 at
    // 7e7 (below, fewer blocks share a compute unit for nothing).
    const bool small = sh.small, wide = n_ub > (int64_t)SB_MAX_BUCKETS * SB_AVG;
    auto launch = g.nf <= 5 ? (small ? sort_launch<8, SB_SMALL_BUCKETS, 2048>
                               : wide ? sort_launch<8, SB_MAX_BUCKETS, 4096> : sort_launch<8, SB_MAX_BUCKETS, 2048>)
                            : (small ? sort_launch<16, SB_SMALL_BUCKETS, 4096> : sort_launch<16, SB_MAX_BUCKETS, 4096>);
    return launch(key_src, r_dst, id_src, id_dst, g, s, sc, sh, n_ub, knew, st);
}
