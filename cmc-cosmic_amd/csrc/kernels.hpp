// Host-side launch entry points of the cmcg kernels (one translation unit per
// phase).  All launches are asynchronous on the given stream; they read the live
// star count from DevScalars on the device, and `n_ub` is only an upper bound used
// to size grids (stars beyond the device-side count exit immediately), so a whole
// step can be enqueued without host round trips.
#pragma once
#include "cmcg_internal.hpp"
#include "mlp.hpp"

// orbit sampler: most LDS samples of any launch variant
constexpr int ORB_MAX_COARSE = 2048;
// sort payload records: at most 16 words (128 B, one cache line) per star
constexpr int SORT_AOS_WORDS = 16;
// The sort's shape: buckets of about SB_AVG stars, at most SB_MAX_BUCKETS (their boundaries
// and counters fill LDS), and the tiles that its count and scatter passes cut the stars
// into.  Up to SB_SMALL_N stars the histogram is small enough for every scatter block to
// sum it, one launch less (at N = 1e5 the whole sort takes 34 us, a launch about 4); there
// a tile is down to one star per thread, for the shortest chain of loads.
constexpr int SB_AVG = 1024, SB_MAX_BUCKETS = 8192, SB_MAX_TILES = 512;
constexpr int64_t SB_SMALL_N = 131072;
constexpr int SB_SMALL_BUCKETS = (int)(SB_SMALL_N / SB_AVG), SB_SMALL_TILES = 32;
struct SortShape { int buckets, tiles; bool small; };
inline SortShape sort_shape(int64_t n_ub)
{
    SortShape sh;
    const int64_t b = (n_ub + SB_AVG - 1) / SB_AVG;
    sh.buckets = b < 1 ? 1 : b > SB_MAX_BUCKETS ? SB_MAX_BUCKETS : (int)b;
    sh.small = n_ub <= SB_SMALL_N;
    const int64_t per = sh.small ? 512 : 2048, most = sh.small ? SB_SMALL_TILES : SB_MAX_TILES;
    const int64_t t = (n_ub + per - 1) / per;
    sh.tiles = t < 1 ? 1 : t > most ? (int)most : (int)t;
    return sh;
}
constexpr uint16_t SB_TAIL = 0xffff;               // bucket number of a star of the SF_INFINITY tail
constexpr uint64_t KEY_INF = 0x8000000000000000ull | 0x4202a05f20000000ull;   // sortable(1.0e10)
__device__ __forceinline__ uint64_t sortable(double x)
{
    uint64_t b = (uint64_t)__double_as_longlong(x);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}
// The step's bucket of a star: its index among the old nodes, cut into B equal parts
// (monotone in the new radius while the old radii ascend).
struct StepBucket {
    double f;
    int B;
    __device__ __forceinline__ StepBucket(int64_t n, int B_) : f((double)B_ / (double)(n + 1)), B(B_) {}
    __device__ __forceinline__ uint32_t operator()(int32_t knew) const
    {
        if (knew < 0) return SB_TAIL;
        const int b = (int)((double)knew * f);
        return b >= B ? B - 1 : b;
    }
};
// Bitonic sort of key[0, S) by the whole block; key holds SMP_MAX words.
constexpr int SMP_MAX = 8192;          // stars sampled for bucket boundaries
__device__ __forceinline__ void sample_sort(uint64_t *key, int S)
{
    int P = 1;
    while (P < S) P <<= 1;
    for (int q = S + threadIdx.x; q < P; q += blockDim.x) key[q] = ~0ull;
    __syncthreads();
    for (int kk = 2; kk <= P; kk <<= 1)
        for (int j = kk >> 1; j > 0; j >>= 1) {
            for (int p = threadIdx.x; p < P / 2; p += blockDim.x) {
                const int q = 2 * p - (p & (j - 1)), x = q | j;       // the p-th pair at distance j
                const uint64_t a = key[q], b = key[x];
                if ((a > b) == ((q & kk) == 0)) { key[q] = b; key[x] = a; }
            }
            __syncthreads();
        }
}

constexpr int RED2_BLOCKS = 64;

constexpr int RIDX_TILE = 4096;     // buckets per block of the radial index's scan
__host__ __device__ constexpr int64_t ridx_entries(int bits) { return ((int64_t)1 << bits) + 2; }
__host__ __device__ constexpr int64_t ridx_tiles(int bits) { return (ridx_entries(bits) + RIDX_TILE - 1) / RIDX_TILE; }

struct Scratch {
    // potential chains
    double *tile_sums;          // two sets of 6 words per tile: estimates, counts, open runs and their prefixes
    int64_t max_tiles;
    double *chain_x;            // chain C's increments
    double *chain_scal;         // 4 doubles
    int64_t *chain_fbad;        // [0]..[2]: a violation in the classification, in the rebuild of B, of C
    int64_t *esa_n;             // [0] sensitive count, [1]..[3] appended counts, [4] the total mass chain's [0]
    // deterministic block partials: 8 doubles per block of the glue, 16 of the orbit sampler
    double *partials;
    int64_t max_blocks;
    // sort
    uint32_t *vals_a;           // sorted permutation: slot of the star now at each position
    uint64_t *sort_split;       // bucket boundaries (order-preserving keys of r), SB_MAX_BUCKETS
    int32_t *sort_moved;        // the general entry point: a star is out of order
    int32_t *sort_uneven;       // the orbit phase's indices do not cut the stars into even buckets (1: its radii do not ascend, 2: counts)
    uint16_t *sort_bkt;         // bucket of every star
    uint32_t *sort_mat;         // tile histograms over the buckets
    size_t sort_mat_cap;
    uint32_t *sort_tot;         // bucket totals
    uint32_t *sort_first;       // first place of every bucket, and the number of stars kept
    uint32_t *sort_order;       // record numbers of buckets beyond the LDS capacity: 2 * sort_aos_cap
    uint64_t *sort_aos;         // packed payload records, SORT_AOS_WORDS words per star
    double2 *mid;               // (r, phi) at every 16th node (search middle level)
    double2 *nodes;             // packed (r, phi) of every node, for the searches
    float2 *pred;               // learned apsides proposals (log r_peri, log r_apo) per star
    uint32_t *ridx;             // radial index: nodes below each bucket of r (ridx_nb + 2 entries)
    uint32_t *ridx_tb;          // its value at every RIDX_TILE-th bucket
    int ridx_bits;              // log2 of the bucket count
    double2 *u_old;             // (new potential, radius), (D, -) at each old sorted radius (set_velocities3)
    double *sv3_dpre;           // D = vold^2 + 2(1-q)(Uoldrold - Uoldrnew) per star, in the order before the step's sort
    unsigned long long *dt_part;  // the step's time step: 64 slots, 128 bytes apart, of complemented dt minima
    double2 *coarse;            // orbit sampler's (r, phi) samples, copied into LDS by every block
    const JumpTables *jump;     // the device's jump tables, shared by its contexts
    double *red2;               // second level of the block-partial reductions (RED2_BLOCKS x 16)
    int64_t sort_aos_cap;
    // set_velocities3 excess chain: per-star excess, ordered event list, per-event
    // walk ends and merge flags, per-block offsets, first failed check
    double *excess_c;
    int64_t *excess_list;
    int64_t *sv3_wend;
    int32_t *sv3_merged;
    int64_t *sv3_blk;
    int64_t *sv3_fallback;      // first presumed head that failed the check
    // tidal stripping loop flag
    int32_t *strip_done;
    // orbit stars deferred to the linear-scan path: KParams::defer_cap entries
    int64_t *defer_list, *defer_kfirst, *defer_order;
    // RNG bases of the current step: [0] relaxation, [1] orbits, [2] orbit slot 1; seeded state
    Rng *rng_base;
    Rng *rng_seeded;
};

hipError_t launch_potential(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub,
                            const Scratch &sc, hipStream_t st, bool count = true);
hipError_t launch_mass_percent(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, const Scratch &sc,
                               const double *pc, int count, int bh_include, double itm, double minimum_r,
                               void *out, void *work, hipStream_t st);
size_t mass_percent_out_bytes();
hipError_t launch_central(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, const Scratch &sc,
                          void *out, void *work, hipStream_t st);
size_t report_work_bytes(const Scratch &sc);     // what both need as `work`
size_t central_out_bytes();
hipError_t launch_potential_at(const DevFields &f, DevScalars *s, const KParams &P,
                               const double *x, double *out, int64_t count, hipStream_t st);

hipError_t launch_sigma(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, hipStream_t st);
hipError_t launch_simul_relax(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, hipStream_t st,
                              bool init_min = true);
hipError_t launch_timestep_sigma(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc,
                                 int64_t n_ub, hipStream_t st);
hipError_t launch_timestep_finalize(DevScalars *s, hipStream_t st);
// threads: block size of the relaxation kernel, one of RELAX_SHAPES (an autotuned
// launch shape; results do not depend on it)
constexpr int RELAX_SHAPES[] = {256, 128, 512, 1024};
constexpr int RELAX_NSHAPES = 4;
hipError_t launch_relax(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc,
                        int64_t n_ub, hipStream_t st,
                        bool with_ec1 = false, int threads = 256);
hipError_t launch_jump_build(const RngTable *T, JumpTables *J, hipStream_t st);
hipError_t launch_rng_bases(DevScalars *s, const Scratch &sc, hipStream_t st);
hipError_t launch_rng_bases_step(DevScalars *s, const Scratch &sc, int64_t step, hipStream_t st);
// the packed node table and the radial index in one pass over r and phi
hipError_t launch_node_index(const DevFields &f, DevScalars *s, const Scratch &sc, int64_t n_ub, int coarse, bool clear,
                             hipStream_t st);
// middle level of the (r, phi) search tables, from the current arrays
hipError_t launch_mid_build(const DevFields &f, DevScalars *s, const Scratch &sc, int64_t n_ub, hipStream_t st);
hipError_t launch_rng_draws(const RngTable *T, const Rng *base, int phase, int64_t first, int64_t count,
                            int ndraw, double *out, hipStream_t st);

// mlp != nullptr: learned brackets (the network's proposals for every star first, on
// the matrix cores, into sc.pred)
hipError_t launch_orbits(const DevFields &f, DevScalars *s, const KParams &P, const RngTable *T,
                         const Scratch &sc, int64_t n_ub, hipStream_t st, const MlpState *mlp = nullptr,
                         float margin = 0.f, hipEvent_t ev_a = nullptr, hipEvent_t ev_b = nullptr, int variant = 0,
                         bool pred_fixed = false, bool index_clear = false);
// proposals equal to the apsides the last orbit phase wrote (log r_peri, log r_apo): a
// perfect predictor, for measuring what any learned proposal could save
hipError_t launch_pred_from_apsides(const DevFields &f, DevScalars *s, const Scratch &sc, int64_t n_ub,
                                    hipStream_t st);
int orbit_variant_count();
void orbit_variant_shape(int v, int *threads, int *coarse, int *cap = nullptr, int *minb = nullptr);
// Device arrays receiving calc_orbit_new's results, one per output.
struct ApsidesOut {
    double *rp, *ra, *dQdrp, *dQdra;
    int64_t *kmin, *kmax;
    int32_t *circular;
};
hipError_t launch_apsides_soa(const DevFields &f, DevScalars *s, const KParams &P, int64_t first, int64_t count,
                              const double *E, const double *J, const ApsidesOut &o, hipStream_t st);
hipError_t launch_find_root_vr(const DevFields &f, DevScalars *s, const KParams &P, int64_t count,
                               const int64_t *j, const int64_t *k, const double *E, const double *J, double *out,
                               hipStream_t st);
hipError_t launch_find_zero_Q(const DevFields &f, DevScalars *s, const KParams &P, int64_t count,
                              const int64_t *j, const int64_t *kmin, const int64_t *kmax,
                              const double *E, const double *J, int64_t *out, hipStream_t st);

hipError_t launch_sort_fields(const double *key_src, double *r_dst, int nf, const uint64_t *const *src,
                              uint64_t *const *dst, DevScalars *s, const Scratch &sc, int64_t n_ub,
                              const int32_t *knew, hipStream_t st);

hipError_t launch_energy_conservation1(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, hipStream_t st);
hipError_t launch_energy_conservation2(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, hipStream_t st,
                                       bool with_ie = false, double *dpre = nullptr, int32_t *strip_done = nullptr,
                                       double *apo_max = nullptr);
constexpr int STRIP_GRAPH_PASSES = 3;     // grid passes of a captured step; a one-block tail kernel finishes rarer longer loops
// the tidal stripping loop: whether one block runs it to its end for a cluster of n_ub stars
bool strip_one_block(int64_t n_ub);
hipError_t launch_strip_loop(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc, bool graph, hipStream_t st,
                             const double *apo_max);
hipError_t launch_strip(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc, int32_t *done,
                        int64_t n_ub, int passes, bool begin, hipStream_t st, const double *apo_max = nullptr);
hipError_t launch_strip_tail(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc, hipStream_t st,
                             const double *apo_max);
hipError_t launch_intermediate_energy(const DevFields &f, DevScalars *s, const KParams &P, int64_t n_ub, hipStream_t st);
hipError_t launch_ie_transfer(const DevFields &f, DevScalars *s, int64_t n_ub, hipStream_t st);
// r_old_sorted: the radii the sort of this step read (old sorted order), or nullptr
hipError_t launch_set_velocities3(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc,
                                  int64_t n_ub, hipStream_t st, const double *r_old_sorted = nullptr,
                                  const double *dpre = nullptr);
hipError_t launch_compute_energy(const DevFields &f, DevScalars *s, const KParams &P, const Scratch &sc,
                                 int64_t n_ub, hipStream_t st, bool end_step = false);

// learned apsides brackets (k_mlp.hip)
int mlp_grid_blocks(int64_t batch);
hipError_t launch_mlp_loss_grad(const MlpState &m, const float *rows, int64_t count, int64_t first, int64_t batch,
                                uint64_t mult, uint64_t off, hipStream_t st);
hipError_t launch_mlp_adam(const MlpState &m, int64_t step, float lr, hipStream_t st);
hipError_t launch_mlp_predict(const MlpState &m, const float *x, int64_t n, float *y, hipStream_t st);
// the network on the matrix cores: every star's proposal (pred[j], j = 1..n), or given rows
hipError_t launch_mlp_infer_stars(const DevFields &f, DevScalars *s, const KParams &P, const MlpState &m,
                                  float2 *pred, int64_t n_ub, hipStream_t st);
hipError_t launch_mlp_infer_rows(const MlpState &m, const float *x, int64_t n, float *y, hipStream_t st);
hipError_t launch_mlp_fit_norm(const MlpState &m, int64_t count, hipStream_t st);
hipError_t launch_mlp_harvest(const DevFields &f, DevScalars *s, const KParams &P, const MlpState &m, int64_t n_ub,
                              hipStream_t st);
