/*
 * step.hip -- the simulation step on CDNA4 (gfx950).
 *
 * A cycle is one launch of bsim_step_kernel: one workgroup per unit of
 * consecutive neurons (a tile or a third of one, layout.h) performs
 *
 *   (ii) phase (ii) of cycle t-1: every synapse into the unit whose pre fired
 *        d cycles earlier adds its weight to the target's E or I accumulator,
 *        in the order the reference's CPU simulator applies them
 *        (src/net/Network.cpp:324-327, src/neuron/lif/LIFENeuron.cpp:52-61);
 *   (i)  the LIF_brian update of cycle t (src/neuron/lif/LIFENeuron.cpp:114-160),
 *        which consumes exactly those accumulators, the spike history update
 *        and the ordered compaction of each 64 neurons' fired bits (by wavefront
 *        ballot) and active (pre, delay) rows, the list that the next launch's
 *        units read.
 *
 * Where a compute unit has more than one unit, one more workgroup orders them
 * for the launches to come, by the work that the launch before recorded
 * (rank_units).
 *
 * A unit finds its active rows from the lists of the blocks of 64 pres that its
 * source chunks cover.  A second launch per cycle, which merged them into one
 * list per 4,096 pres, took 4 us of a cycle of a few dozen neurons and 8 to 11
 * of large ones, with the launch's own start: us per cycle with it and without,
 * 48 neurons 11.3 / 7.7, 9,896 10.8 / 7.8, 230,000 in 96 chains 33.0 / 28.5,
 * 330,000 63.2 / 61.4, 650,000 113 / 111.
 *
 * Phase (ii) for a unit: the sub-rows of its active rows, in list order, form
 * one stream of events, which the workgroup takes in passes of PASS = 1,024
 * positions.  The NEV event wavefronts find each position's synapse and load
 * it, and sort the pass by target, keeping stream order (event_wave); the NOWN
 * owner wavefronts, whose threads hold the targets' E and I accumulators in
 * registers, add a pass's events while the event wavefronts prepare the next
 * (owner_wave), and update the targets in the end (update_unit).  The two kinds
 * of wavefront have no code in common from the workgroup's first batch to its
 * end (event_unit, owner_unit): with one body for both, branching at each
 * phase, the compiler kept the state of either alive in the other, 69 vector
 * registers and no room to load anything early, against 52; us per cycle of
 * 48 neurons 8.2 / 7.2, 9,896 9.1 / 7.2, 330,000 61.3 / 59.9, a sweep of
 * 300 chains 45.2 / 42.4.  Every accumulator thus receives its adds one at a time in
 * stream order, (pre, delay, creation) -- the creation order the host
 * verified -- so the sums are the reference's sequential fp32 sums, bit for
 * bit, with no floating-point atomics.
 *
 * What bounds it: a unit is a chain of passes, each a chain of LDS round trips,
 * a barrier and the synapse loads, so the launch is as long as its longest
 * unit, or the units' time over the 512 workgroups that fit at a time (two per
 * compute unit).  Where the parallelism of a unit comes from decides that: one
 * wavefront per part that walked every row, expanded its own sub-rows and
 * applied them by masks per 64 events took 3.8 us per 768 events; here the
 * expansion and the sort of 1,024 events are spread over eight wavefronts,
 * every row is expanded once and not once per part, and the sequential part,
 * the adds, is left to the owners: 2 us.  Whole step launch, before and now:
 * 330,000 neurons at ~100 Hz (3.1e6 events) 83 / 54 us, 110,000 at ~1,600 Hz
 * with delays up to 50 steps (3.2e7 events) 3,408 / 877, 96 chains of 100 to
 * 1,000 neurons (2.4e5 events) 46 / 29, 650,000 neurons at ~100 Hz (7e6
 * events, workgroups of eight wavefronts) 106 / 91.  Measured and not used: 4
 * event wavefronts for all but the last (71, 1,930, 33 us when these took 60, 927
 * and 30), 16 (one workgroup per compute unit), LDS masks by target instead of
 * ballots (70 against 60 us for the first), four wavefronts that each take the
 * add of their own targets (71).
 *
 * Arithmetic: compiled with -ffp-contract=off (no FMA contraction) and
 * without denormal flushing, so V = ((Cm*V + v_tmp) + iE*C_E) + iI*C_I rounds
 * exactly as the reference's CPU code.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "layout.h"

#define WAVE 64
#ifndef NEV                           /* step_many.hip sets it and STEP_EU */
#define NEV 8                         /* event wavefronts of a step workgroup */
#define STEP_EU 6                     /* wavefronts per SIMD: two workgroups per compute unit */
#endif
#define NOWN 4                        /* owner wavefronts */
#define NTHREAD (WAVE * (NEV + NOWN))
#define NCOL 16                       /* groups of 64 events in a pass */
#define PASS (NCOL * WAVE)
#define NGRP (NCOL / NEV)             /* groups of an event wavefront */
#define NO_MARK 0xFFFFFFFFu           /* no synapse index: a group has fewer than 2^32 - 1 */
#define MAXR 32                       /* source chunks per batch */
#define BLKS (BSIM_CHUNK / WAVE)      /* blocks of 64 pres per source chunk */
#define NRES 8                        /* XCDs: workgroup w runs on XCD (w + c) mod 8 */
static_assert(BLKS == WAVE, "a lane per block of a source chunk");
static_assert(NCOL == 16 && NCOL % NEV == 0, "a target's histogram row is one 16-byte vector");

/* Slots per target: a pass puts PASS / U events on a target of a unit of U on
 * average, if full; three times that, at least 8. */
__host__ __device__ static constexpr uint32_t slots_of(uint32_t U)
{
    return U >= 384 ? 8u : (3u * PASS / U) & ~3u;
}

/* LDS bytes of a workgroup: chunk | hist | mark | slot | blk_end | blk_mark | btot, ctot, most, last */
__host__ __device__ static constexpr size_t lds_bytes(uint32_t U)
{
    return 16 * MAXR + 2 * U * NCOL + 8 * PASS + 4 * slots_of(U) * U + 4 * MAXR * BLKS + 4 * NEV * WAVE + 8 * NEV +
           8 * MAXR + 16;
}

__device__ __forceinline__ uint32_t bern_hash(uint64_t seed, uint32_t id, uint32_t t)
{
    uint64_t z = seed ^ (((uint64_t)id << 32) | (uint64_t)t);
    z += 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (uint32_t)(z >> 32);
}

/* X ~ Poisson from the uniform u by binary search of the rate's inverse-CDF
 * table (layout.h) */
__device__ __forceinline__ uint32_t poisson_pick(const uint32_t *tab, uint32_t u)
{
    uint32_t lo = 0, hi = tab[0] - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (u < tab[1 + mid]) hi = mid; else lo = mid + 1;
    }
    return lo;
}

__device__ __forceinline__ uint64_t ballot64(bool p) { return __builtin_amdgcn_ballot_w64(p); }

__device__ __forceinline__ uint32_t readlane(uint32_t x, int32_t l)
{
    return __builtin_amdgcn_readlane(x, l);
}

/* A value that is the same in every lane (an LDS word all lanes read, the
 * wavefront index), moved to a scalar register: branches and loops on it are
 * then scalar branches, not exec-masked ones.  Without this the compiler
 * cannot tell that such a loop exits at once for the whole wavefront; it
 * builds the loop with lane masks, merges its exit paths, and waits for all
 * loads in flight where the paths join. */
__device__ __forceinline__ uint32_t uniform(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ uint32_t wave_index() { return uniform(threadIdx.x / WAVE); }

/* DPP controls (GFX9 encoding): shift right within a row of 16 lanes, and
 * broadcast lane 15 / 31 into the following rows */
#define DPP_ROW_SHR(n) (0x110 + (n))
#define DPP_ROW_BCAST15 0x142
#define DPP_ROW_BCAST31 0x143

/* The device clock: the cycle of the coming clocked step launch.  Every
 * workgroup of a clocked launch adds one to the completion counter of its XCD
 * residue x = workgroup % 8 when it ends (an atomic whose result nobody waits
 * for); each residue holds 1 / 8 of the grid, so its counter grows by that
 * much per launch.  While any workgroup of launch t runs, its own residue's
 * counter lies in [t grid / 8, (t + 1) grid / 8) -- it has not added its one
 * yet -- so the quotient is t.  Plain (scalar,
 * cached) loads: a launch sees the counts of the launches before it, and a
 * value cached during the launch is still within its interval.  (A single
 * counter whose last incrementer advanced the cycle made every workgroup wait
 * on one contended address: 48 against 20 us per launch in a cycle without
 * deliveries.) */
__device__ __forceinline__ int32_t device_cycle(const bsim_dev &d, uint32_t x)
{
    /* count / (grid / 8) without an integer division: the quotient's
     * fractional part is a multiple of 8 / grid, so half of that added
     * before truncation absorbs the rounding of the product (below 2^-20 for
     * cycles below 2^31, against a half step of at least 2^-19 for grids of
     * up to 2^18 workgroups per residue) */
    const double c = (double)d.done[BSIM_DONE_STRIDE * x];
    return (int32_t)(c * d.done_inv + 0.5 * d.done_inv);
}

/* inclusive prefix sum over the wavefront: four in-row shifts, then the row
 * totals are carried across rows by two broadcasts; lanes without a source
 * read 0 */
__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t x)
{
    int v = (int)x;
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(1), 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(2), 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(4), 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_SHR(8), 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_BCAST15, 0xa, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, DPP_ROW_BCAST31, 0xc, 0xf, false);
    return (uint32_t)v;
}

/* ---- delivery ------------------------------------------------------------- */

/* A source chunk of the batch: where its row table starts in off_tab (low and
 * high word), its first block of 64 pres, table entries per row. */
struct __attribute__((aligned(16))) Chunk {
    uint32_t ob_lo, ob_hi, blk, st;
};

struct Shared {
    Chunk *chunk;               /* [MAXR] */
    uint32_t *hist;             /* [2][U][NCOL / 4] events of each target per group, one byte each */
    uint32_t *mark;             /* [2][PASS] synapse index where a sub-row or group starts, else NO_MARK */
    float *slot;                /* [K][U] a pass's weights of each target in stream order */
    uint32_t *blk_end;          /* [MAXR][BLKS] active rows of a chunk up to the end of each of its blocks */
    uint32_t *blk_mark;         /* [NEV][64] first rows of blocks among 64 rows (load_entries), else NO_MARK */
    uint32_t *btot;             /* [2][NEV] stream length of each event wavefront's rows of a block */
    uint32_t *ctot;             /* [2][MAXR] active rows of each chunk */
    uint32_t *most;             /* [2] largest rank of a pass's events beyond the slots */
    uint32_t *last;             /* [2] the pass is the batch's last */
};

/* orders this wavefront's LDS accesses (lanes exchange data through LDS) */
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ void wg_barrier() { __syncthreads(); }

/* The batch's active rows: those of its chunks in order, of a chunk's blocks of
 * 64 pres in order, of a block as its list has them.  Lane c < nrb holds the
 * rows up to the end of chunk c; at: the chunk that the next rows start in. */
struct Rows {
    uint32_t end;
    int32_t nrb, at;
};

__device__ __forceinline__ uint32_t chunk_end(const Rows &R, int32_t c) { return c < 0 ? 0u : readlane(R.end, c); }

/* List entries of WR times 64 rows (lane l: rows l, 64 + l, ...): e = (p % 64)
 * << 6 | d - 1 of the row, cb = chunk << 6 | block of its pre. */
template <int WR>
struct Entries {
    uint32_t e[WR], cb[WR];
    uint32_t n;                 /* rows (uniform) */
};

/* Loads the list entries of the rows from j0 on.  Every block that has any of
 * 64 of them marks its first (with the block, and how many of its rows come
 * before); a row's block is that of the last mark at or before it. */
template <int WR>
__device__ __forceinline__ void load_entries(const Shared &S, const bsim_dev &d, const uint16_t *seg, Rows &R,
                                             uint32_t j0, uint32_t nrows, Entries<WR> &E)
{
    E.n = j0 < nrows ? min((uint32_t)(WR * WAVE), nrows - j0) : 0u;
    const uint32_t lane = threadIdx.x & (WAVE - 1), cap = WAVE * (uint32_t)d.dmax;
    uint32_t *mk = S.blk_mark + wave_index() * WAVE;
#pragma unroll
    for (int i = 0; i < WR; i++) {
        if (E.n <= (uint32_t)(i * WAVE)) continue;            /* uniform */
        const uint32_t b = j0 + i * WAVE, e1 = b + min((uint32_t)WAVE, E.n - i * WAVE);
        while (chunk_end(R, R.at) <= b) R.at++;
        for (int32_t c = R.at;; c++) {
            const uint32_t base = chunk_end(R, c - 1), ce = chunk_end(R, c);
            const uint32_t e = base + S.blk_end[c * BLKS + lane];
            const uint32_t s = lane > 0 ? base + S.blk_end[c * BLKS + lane - 1] : base;
            const uint32_t lo = max(s, b), hi = min(e, e1);
            if (hi > lo) mk[lo - b] = (uint32_t)c << 6 | lane | (lo - s) << 11;
            if (ce >= e1) break;
        }
        wave_sync();
        const uint32_t v = mk[lane];
        mk[lane] = NO_MARK;
        wave_sync();
        const uint64_t m = ballot64(v != NO_MARK) & (~0ull >> (WAVE - 1 - lane));
        const uint32_t at = (WAVE - 1) - (uint32_t)__clzll((long long)(m | 1ull));
        const uint32_t f = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(at * 4u), (int)v);
        E.cb[i] = f & (MAXR * BLKS - 1);
        /* lanes past the last row load an entry of its block's list */
        const uint32_t x = min((f >> 11) + lane - at, cap - 1u);
        E.e[i] = seg[(uint64_t)(S.chunk[E.cb[i] >> 6].blk + (E.cb[i] & 63u)) * cap + x];
    }
}

typedef uint32_t pair_u32 __attribute__((ext_vector_type(2), aligned(4)));

/* Loads the rows' table entries: each sub-row's start and the start of the one
 * after it. */
template <int WR>
__device__ __forceinline__ void load_rows(const Shared &S, const bsim_dev &d, const Entries<WR> &E, pair_u32 (&ab)[WR])
{
#pragma unroll
    for (int i = 0; i < WR; i++) {
        if (E.n <= (uint32_t)(i * WAVE)) continue;            /* uniform */
        const uint4 ch = *reinterpret_cast<const uint4 *>(S.chunk + (E.cb[i] >> 6));
        /* an entry past the end of its block's list is any word: kept within the
         * block's rows */
        const uint32_t row = ((E.cb[i] & 63u) * WAVE + (E.e[i] >> 6 & 63u)) * (uint32_t)d.dmax +
                             min(E.e[i] & 63u, (uint32_t)d.dmax - 1u);
        ab[i] = *reinterpret_cast<const pair_u32 *>(d.off_tab + ((uint64_t)ch.y << 32 | ch.x) + (uint64_t)(row * ch.w));
    }
}

/* A block of NEV * 64 * WR rows, WR per thread of the event wavefronts: the row's
 * sub-row into the unit as its first synapse, its length and its position in
 * the batch's stream of events. */
template <int WR>
struct Block {
    uint32_t a[WR], len[WR], pos[WR];
};

/* The block's sub-rows from its table entries (n rows in this wavefront), with
 * positions within the wavefront; the wavefront's stream length goes to btot. */
template <int WR>
__device__ __forceinline__ void make_block(const Shared &S, const pair_u32 (&ab)[WR], uint32_t n, uint32_t buf,
                                           Block<WR> &k)
{
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    uint32_t at = 0;
#pragma unroll
    for (int i = 0; i < WR; i++) {
        k.a[i] = ab[i].x;
        k.len[i] = i * WAVE + lane < n ? ab[i].y - ab[i].x : 0u;
        const uint32_t incl = wave_incl_scan(k.len[i]);
        k.pos[i] = at + incl - k.len[i];
        at += readlane(incl, WAVE - 1);
    }
    if (lane == 0) S.btot[buf * NEV + wave_index()] = at;
}

/* Positions in the batch's stream, once every wavefront has written btot: at is
 * the stream's length so far (uniform), advanced past the block. */
template <int WR>
__device__ __forceinline__ void place_block(const Shared &S, uint32_t buf, Block<WR> &k, uint32_t &at)
{
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    const uint32_t incl = wave_incl_scan(lane < NEV ? S.btot[buf * NEV + lane] : 0u);
    const uint32_t w = wave_index(), before = at + (w > 0 ? readlane(incl, (int32_t)w - 1) : 0u);
#pragma unroll
    for (int i = 0; i < WR; i++) k.pos[i] += before;
    at += readlane(incl, WAVE - 1);
}

/* The events of a pass, stream positions [b, e) with e - b <= PASS: event
 * wavefront w takes the groups of 64 positions w, w + NEV, ...  Each sub-row
 * marks its first position in the pass, and every multiple of 64 that it
 * covers, with the synapse index there (put_marks); a position's synapse lies
 * past the last mark at or before it in its group, the highest set bit of the
 * group's ballot (load_events). */
template <int WR>
__device__ __forceinline__ void put_marks(uint32_t *mark, const Block<WR> &k, uint32_t b, uint32_t e)
{
#pragma unroll
    for (int i = 0; i < WR; i++) {
        const uint32_t lo = max(k.pos[i], b), hi = min(k.pos[i] + k.len[i], e);
        if (hi > lo) {
            const uint32_t x = lo - b, y = hi - b, a = k.a[i] + (lo - k.pos[i]);
            mark[x] = a;
            for (uint32_t g = (x | (WAVE - 1)) + 1u; g < y; g += WAVE) mark[g] = a + (g - x);
        }
    }
}

struct Step {
    uint32_t tgt[NGRP];
    float w[NGRP];
};

__device__ __forceinline__ void load_events(uint32_t *mark, const bsim_syn *syn, uint32_t nsyn, Step &st)
{
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    const uint64_t le = ~0ull >> (WAVE - 1 - lane);           /* bits 0..lane */
    uint32_t *mk = mark + wave_index() * WAVE + lane;
    uint32_t v[NGRP], at[NGRP];
#pragma unroll
    for (int g = 0; g < NGRP; g++) v[g] = mk[g * NEV * WAVE];
#pragma unroll
    for (int g = 0; g < NGRP; g++) mk[g * NEV * WAVE] = NO_MARK;
#pragma unroll
    for (int g = 0; g < NGRP; g++) {
        const uint64_t m = ballot64(v[g] != NO_MARK) & le;
        at[g] = (WAVE - 1) - (uint32_t)__clzll((long long)(m | 1ull));
    }
#pragma unroll
    for (int g = 0; g < NGRP; g++) v[g] = (uint32_t)__builtin_amdgcn_ds_bpermute((int)(at[g] * 4u), (int)v[g]);
#pragma unroll
    for (int g = 0; g < NGRP; g++) {
        /* lanes past the pass's end load some synapse of the group */
        uint32_t addr = v[g] + (lane - at[g]);
        if (addr >= nsyn) addr = 0u;
        const bsim_syn sv = syn[addr];
        st.tgt[g] = sv.tgt;
        st.w[g] = __uint_as_float(sv.w);
    }
}

/* The lanes whose NB-bit value x equals this lane's, among the lanes in v. */
template <int NB>
__device__ __forceinline__ uint64_t same_lanes(uint32_t x, uint64_t v)
{
    const uint32_t nx = ~x;
    uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int32_t z = __builtin_amdgcn_sbfe((int32_t)nx, b, 1);   /* 0 where the bit is set, else -1 */
        const uint64_t B = ballot64(z == 0);
        lo &= (uint32_t)B ^ (uint32_t)z;
        hi &= (uint32_t)(B >> 32) ^ (uint32_t)z;
    }
    return (uint64_t)lo | ((uint64_t)hi << 32);
}

__device__ __forceinline__ uint32_t byte_sum(uint32_t x, uint32_t acc) { return __builtin_amdgcn_sad_u8(x, 0u, acc); }

/* Event wavefronts: phase (ii) of one batch of nrows active rows.  A pass adds
 * up to PASS events, in stream order, to their targets' accumulators:
 *   count    per group of 64 events, a target's first event finds the others of
 *            its target by ballots and stores how many there are in the group's
 *            byte of the target's histogram row;
 *   place    an event's rank among its target's events of the pass is the sum
 *            of the bytes of the groups before its own plus the events of its
 *            target in the lanes below; its weight goes to the target's slot
 *            of that rank;
 *   add      (owner wavefronts, while these count the next pass) every target's
 *            owner adds its slots in order.
 * A target with more events than slots takes further rounds of place and add.
 * The loads run ahead of the passes: a pass's synapses are loaded during the
 * pass before, the table entries and list entries one and two blocks ahead of
 * the rows that the marks are put from. */
template <int NB, int WR>
__device__ void event_wave(const Shared &S, const bsim_dev &d, uint32_t qoff, uint32_t nsyn, Rows &R, uint32_t nrows,
                           const uint16_t *seg, uint32_t U, uint32_t K, uint32_t &par, const bsim_syn *syn, uint32_t &events)
{
    const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1), w = wave_index();
    const uint64_t lt = (1ull << lane) - 1ull;
    constexpr uint32_t BROWS = NEV * WAVE * WR; /* rows of a block */
    uint32_t jn = w * (WR * WAVE);                     /* first row of the next block to look up */
    Entries<WR> E;
    pair_u32 ab[WR];
    Block<WR> k0, k1;                               /* blocks not yet used up */
    uint32_t e0 = 0, e1 = 0, at = 0;            /* ends of k0, k1 and of the stream so far */
    uint32_t q = 1, buf = 0;                    /* how many of k0, k1 are in use */
    uint32_t left = nrows > BROWS ? nrows - BROWS : 0u;    /* rows past the blocks made */
    Step X;
    load_entries(S, d, seg, R, jn, nrows, E);
    uint32_t nab = E.n;
    load_rows(S, d, E, ab);
    load_entries(S, d, seg, R, jn += BROWS, nrows, E);
    make_block(S, ab, nab, 0u, k0);
    nab = E.n;
    load_rows(S, d, E, ab);
    load_entries(S, d, seg, R, jn += BROWS, nrows, E);
    if (left > 0) {                                           /* uniform */
        make_block(S, ab, nab, buf = 1u, k1);
        nab = E.n;
        load_rows(S, d, E, ab);
        load_entries(S, d, seg, R, jn += BROWS, nrows, E);
        left = left > BROWS ? left - BROWS : 0u;
        q = 2;
    }
    wg_barrier();
    place_block(S, 0u, k0, at);
    e0 = at;
    if (q == 2) {
        place_block(S, 1u, k1, at);
        e1 = at;
    }
    uint32_t b = 0, n = min(at, (uint32_t)PASS);              /* the pass: n events from position b */
    uint32_t *mark = S.mark;                                  /* the coming pass's marks */
    put_marks(mark, k0, 0u, n);
    if (q == 2) put_marks(mark, k1, 0u, n);
    while (q > 0 && n >= e0) {
        k0 = k1;
        e0 = e1;
        q--;
    }
    wg_barrier();
    load_events(mark, syn, nsyn, X);
    while (true) {
        /* a wavefront may put the next pass's marks while another still reads this one's */
        mark = mark == S.mark ? S.mark + PASS : S.mark;
        uint32_t li[NGRP], rk[NGRP];
        float wt[NGRP];
#pragma unroll
        for (int g = 0; g < NGRP; g++) {
            li[g] = X.tgt[g] - qoff;
            wt[g] = X.w[g];
        }
        /* the next pass and the block after the ones in use.  No load is in
         * flight here, and the conditional ones follow one another without a
         * wait in between: the wait counter is in order, and the compiler
         * waits for every load that it cannot count */
        const uint32_t nb = b + n;
        const uint32_t nn = min((q == 2 ? e1 : q == 1 ? e0 : nb) - nb, (uint32_t)PASS);
        if (q > 0) put_marks(mark, k0, nb, nb + nn);
        if (q > 1) put_marks(mark, k1, nb, nb + nn);
        while (q > 0 && nb + nn >= e0) {
            k0 = k1;
            e0 = e1;
            q--;
        }
        const bool more = q < 2 && left > 0;
        Block<WR> kn;
        if (more) {
            make_block(S, ab, nab, buf ^= 1u, kn);
            nab = E.n;
            load_rows(S, d, E, ab);
            load_entries(S, d, seg, R, jn += BROWS, nrows, E);
            left = left > BROWS ? left - BROWS : 0u;
        }
        uint32_t *hist = S.hist + par * (U * (NCOL / 4));
#pragma unroll
        for (int g = 0; g < NGRP; g++) {
            const uint32_t col = w + g * NEV;                 /* uniform */
            rk[g] = 0u;
            if (col * WAVE < n) {                             /* uniform */
                const bool v = col * WAVE + lane < n;
                if (!v) li[g] = 0u;
                const uint64_t m = same_lanes<NB>(li[g], ballot64(v));
                rk[g] = (uint32_t)__popcll(m & lt);
                if (v && rk[g] == 0u)
                    reinterpret_cast<uint8_t *>(hist)[li[g] * NCOL + col] = (uint8_t)__popcll(m);
            }
        }
        wg_barrier();
        if (more) {
            place_block(S, buf, kn, at);
            if (q == 0) {
                k0 = kn;
                e0 = at;
            } else {
                k1 = kn;
                e1 = at;
            }
            q++;
        }
        const bool done = nn == 0 && q == 0 && left == 0;     /* uniform */
        if (!done) load_events(mark, syn, nsyn, X);
        uint32_t over = 0u;             /* largest rank beyond the slots */
#pragma unroll
        for (int g = 0; g < NGRP; g++) {
            const uint32_t col = w + g * NEV;                 /* uniform */
            if (col * WAVE < n) {                             /* uniform */
                const bool v = col * WAVE + lane < n;
                const uint4 h = reinterpret_cast<const uint4 *>(hist)[li[g]];
                const uint32_t x = col / 4, mask = (1u << (8u * (col % 4))) - 1u;
                uint32_t r = rk[g];
                r = byte_sum(h.x & (x > 0 ? ~0u : mask), r);
                r = byte_sum(h.y & (x > 1 ? ~0u : x == 1 ? mask : 0u), r);
                r = byte_sum(h.z & (x > 2 ? ~0u : x == 2 ? mask : 0u), r);
                r = byte_sum(h.w & (x == 3 ? mask : 0u), r);
                rk[g] = r;
                if (v && r < K) S.slot[r * U + li[g]] = wt[g];
                if (v && r >= K) over = max(over, r);
            }
        }
        if (over) atomicMax(&S.most[par], over);
        if (tid == 0) {
            S.most[par ^ 1u] = 0u;
            S.last[par] = done ? 1u : 0u;
        }
        wg_barrier();
        for (uint32_t r0 = K, most = uniform(S.most[par]); most >= r0; r0 += K) {
            wg_barrier();
#pragma unroll
            for (int g = 0; g < NGRP; g++)
                if ((w + g * NEV) * WAVE + lane < n && rk[g] - r0 < K)
                    S.slot[(rk[g] - r0) * U + li[g]] = wt[g];
            wg_barrier();
        }
        par ^= 1u;
        if (done) break;
        b = nb;
        n = nn;
    }
    events += at;
}

/* E and I accumulators of an owner thread's targets: o, o + NOWN * 64, ... of
 * the unit, o its index among the owner threads. */
template <int S_>
struct Acc {
    float e[S_], i[S_];
};

/* Owner wavefronts: the passes of one batch. */
template <int S_>
__device__ void owner_wave(const Shared &S, uint32_t U, uint32_t K, uint32_t &par, Acc<S_> &acc)
{
    const uint32_t o = threadIdx.x - NEV * WAVE;
    wg_barrier();
    wg_barrier();
    while (true) {
        wg_barrier();
        wg_barrier();
        const uint32_t most = uniform(S.most[par]), last = uniform(S.last[par]);
        uint32_t *hist = S.hist + par * (U * (NCOL / 4));
        uint32_t tot[S_];
        for (uint32_t r0 = 0;; r0 += K) {
#pragma unroll
            for (int j = 0; j < S_; j++) {
                const uint32_t i = o + j * (NOWN * WAVE);
                if (uniform(i) >= U) continue;                /* U is whole wavefronts */
                /* a slot past the target's events counts as 0: the sums, which
                 * start at +0 and never become -0, do not change by it */
                const float *sl = S.slot + i;
                float x[4];
#pragma unroll
                for (uint32_t y = 0; y < 4; y++) x[y] = sl[y * U];
                if (r0 == 0) {                                /* uniform */
                    const uint4 h = reinterpret_cast<const uint4 *>(hist)[i];
                    reinterpret_cast<uint4 *>(hist)[i] = make_uint4(0u, 0u, 0u, 0u);
                    tot[j] = byte_sum(h.x, byte_sum(h.y, byte_sum(h.z, byte_sum(h.w, 0u))));
                }
                const uint32_t n = min(tot[j] > r0 ? tot[j] - r0 : 0u, K);
                uint32_t r = 0;
                while (true) {
                    float z[4];
#pragma unroll
                    for (uint32_t y = 0; y < 4; y++) z[y] = x[y];
                    const bool go = ballot64(r + 4 < n) != 0ull;              /* uniform; then r + 4 < K */
                    if (go) {
#pragma unroll
                        for (uint32_t y = 0; y < 4; y++) x[y] = sl[(r + 4 + y) * U];
                    }
#pragma unroll
                    for (uint32_t y = 0; y < 4; y++) {
                        const float a = r + y < n ? z[y] : 0.0f;
                        acc.e[j] += a >= 0.0f ? a : 0.0f;
                        acc.i[j] += a >= 0.0f ? 0.0f : a;
                    }
                    if (!go) break;
                    r += 4;
                }
            }
            if (most < r0 + K) break;                         /* uniform */
            wg_barrier();
            wg_barrier();
        }
        par ^= 1u;
        if (last) break;
    }
}

/* Event wavefronts: where the batch's source chunks lie and how many active
 * rows each of their blocks has, one chunk at a time each.  The first
 * BSIM_UNIT_CHUNKS of a unit are in its record. */
__device__ __forceinline__ void prepare_batch(const Shared &S, const bsim_dev &d, const bsim_unit *un, int32_t rb,
                                              int32_t nrb, int32_t list, uint32_t buf)
{
    uint32_t lane = threadIdx.x & (WAVE - 1);
#ifdef STEP_MANY
    /* keeps the addresses below from being held in registers from batch to batch,
     * where the one too many went to private memory */
    asm volatile("" : "+v"(lane));
#endif
    const uint32_t *cnt = d.seg_count + (int64_t)list * d.nwords;
    for (int32_t c = (int32_t)wave_index(); c < nrb; c += NEV) {
        uint64_t ob;
        uint32_t blk, nblk, st;
        if (rb + c < BSIM_UNIT_CHUNKS) {
            const bsim_chunk h = un->chunk[rb + c];
            ob = (uint64_t)h.off_base;
            blk = h.blk;
            nblk = h.nblk;
            st = h.stride;
        } else {
            const bsim_range r = d.rng[un->rng0 + rb + c];
            ob = (uint64_t)r.off_base + (uint64_t)un->part;
            blk = (uint32_t)r.lo / WAVE;
            nblk = (uint32_t)(r.hi - r.lo) / WAVE;
            st = r.stride;
        }
        const uint32_t incl = wave_incl_scan(lane < nblk ? cnt[blk + lane] : 0u);
        S.blk_end[c * BLKS + lane] = incl;
        if (lane == WAVE - 1) {
            S.ctot[buf * MAXR + c] = incl;
            S.chunk[c] = Chunk{(uint32_t)ob, (uint32_t)(ob >> 32), blk, st};
        }
    }
}

/* The state of an owner thread's neurons that phase (i) reads, loaded
 * before phase (ii) so that its latency is hidden behind the delivery (no
 * other workgroup writes these words during the launch: a neuron belongs to
 * one unit, and the history words read are the previous cycle's copy).  Kept
 * in registers up to PREFETCH_MAX_S slots per lane. */
#ifndef PREFETCH_MAX_S
#define PREFETCH_MAX_S 1
#endif
template <int S_>
struct NState {
    uint32_t cls[S_];
    int32_t refrac[S_];
    float v[S_], ie[S_], ii[S_], vtmp[S_];
    uint64_t hist[S_];
    bsim_lifc c[S_];
};

template <int S_>
__device__ __forceinline__ void load_nstate(const bsim_dev &d, int32_t base, const uint64_t *hist_in,
                                            NState<S_> &ns)
{
#pragma unroll
    for (int j = 0; j < S_; j++) {
        const int32_t nid = base + j * (NOWN * WAVE) + (int32_t)threadIdx.x - NEV * WAVE;
        const bool valid = nid < d.n;
        const int32_t x = valid ? nid : 0;
        ns.cls[j] = d.ncls[x];
        ns.refrac[j] = d.refrac[x];
        ns.v[j] = d.v[x];
        ns.ie[j] = d.ie[x];
        ns.ii[j] = d.ii[x];
        ns.vtmp[j] = d.v_tmp[x];
        ns.hist[j] = hist_in[x];
    }
}

/* The neurons' parameter sets, once their classes have arrived. */
template <int S_>
__device__ __forceinline__ void load_params(const bsim_dev &d, NState<S_> &ns)
{
#pragma unroll
    for (int j = 0; j < S_; j++)
        ns.c[j] = d.lifc[ns.cls[j] >> 30 == BSIM_KIND_LIF ? ns.cls[j] & BSIM_CLS_SET_MASK : 0u];
}

/* This workgroup of a clocked launch has ended its cycles (see device_cycle). */
__device__ __forceinline__ void count_done(const bsim_dev &d, uint64_t cycles)
{
    (void)__hip_atomic_fetch_add(d.done + BSIM_DONE_STRIDE * (blockIdx.x % 8u), cycles, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
}

/* Orders the units for the coming launches by their work in the launch before
 * (results do not depend on the order; the firing volleys move slowly against
 * two cycles).  The hardware deals the workgroups out to the XCDs in turn, slot s
 * to XCD s % 8, and starts an XCD's in order.  The units are cut, in index order,
 * into eight runs of equal cost, one per XCD: units of a group, which read the
 * same rows at the same time, so share an L2.  An XCD has slots for an eighth of
 * the units; the lightest of a longer run fill what others leave free, so that no
 * XCD starts more workgroups than another.  us per cycle with whole groups on XCDs
 * / with the units dealt out in turn where those were uneven / with runs: 330,000
 * neurons at ~100 Hz 59.9 / 54.5 / 55.0, 650,000 108 / 101 / 98.9, 110,000 with
 * delays up to 50 steps 950 / 1,046 / 877, a sweep of 96 chains 27.6 / 27.9 /
 * 27.1, the same in units of half the size 21.7 / 21.9 / 21.2.  Twice the slots,
 * so that runs stay whole: 59.5, 110, 875, 26.9, 22.9 (XCDs with few heavy units
 * start more).
 *
 * Within an XCD the heavy units come first, by half-octave classes (counting
 * sort).  Within a class the order is arbitrary up to delays of RANK_ORDERED_DMAX
 * steps, and while two workgroups per compute unit hold all units; past them,
 * where most lines are row-table entries that a group's units share while they
 * run together, units keep their order: 1,010,000 neurons with delays up to 50
 * steps 7.65 / 6.14 ms, 410,000 2.51 / 2.36, but 330,000 with delays up to 6 56.5
 * / 57.9 us.
 *
 * Runs in one workgroup, beside the others of the launch, and clears the loads
 * that it has read.  The classes of the units are kept in LDS where they fit. */
#define RANK_CLASSES 64
#define RANK_FIXED 8192ull
#define RANK_ORDERED_DMAX 24

__device__ __forceinline__ uint32_t load_class(uint64_t x)
{
    if (x < 16) return 0;
    const uint32_t e = 63u - (uint32_t)__builtin_clzll(x);        /* floor(log2 x) >= 4 */
    const uint32_t h = (uint32_t)(x >> (e - 1)) & 1u;              /* next bit */
    return min(2u * (e - 4u) + h + 1u, (uint32_t)RANK_CLASSES - 1u);
}

/* The cost of a unit of class c: its work, and that of a workgroup that finds
 * next to nothing to deliver. */
__device__ __forceinline__ uint64_t class_cost(uint32_t c)
{
    return RANK_FIXED + (c == 0 ? 0ull : (2ull + ((c - 1u) & 1u)) << ((c - 1u) / 2u + 3u));
}

__device__ void rank_units(const bsim_dev &d, uint64_t *load, int32_t *perm, uint32_t *lds, uint32_t lds_size)
{
    uint64_t *sum = reinterpret_cast<uint64_t *>(lds);              /* [NTHREAD] */
    uint32_t *cnt = reinterpret_cast<uint32_t *>(sum + NTHREAD), *fill = cnt + NRES * RANK_CLASSES;
    uint32_t *rtot = fill + NRES * RANK_CLASSES;                    /* [NRES] */
    uint8_t *cls = (uint32_t)d.ntiles <= lds_size - (8u * NTHREAD + 4u * (2 * NRES * RANK_CLASSES + NRES))
                       ? reinterpret_cast<uint8_t *>(rtot + NRES) : d.tile_cls;
    static_assert(RANK_CLASSES == WAVE && NRES * RANK_CLASSES <= NTHREAD, "a wavefront per residue, a lane per class");
    const uint32_t tid = threadIdx.x;
    const bool counts = tid < NRES * RANK_CLASSES;
    if (counts) cnt[tid] = 0u;
    /* thread: units k0 .. k1 - 1 */
    const int32_t per = (d.ntiles + NTHREAD - 1) / NTHREAD;
    const int32_t k0 = min((int32_t)tid * per, d.ntiles), k1 = min(k0 + per, d.ntiles);
    uint64_t mine = 0;
    for (int32_t k = k0; k < k1; k++) {
        const uint32_t c = load_class(load[k]);
        load[k] = 0ull;
        cls[k] = (uint8_t)c;
        mine += class_cost(c);
    }
    uint64_t upto = mine;
    for (uint32_t o = 1; o < NTHREAD; o <<= 1) {
        sum[tid] = upto;
        __syncthreads();
        if (tid >= o) upto += sum[tid - o];
        __syncthreads();
    }
    sum[tid] = upto;
    __syncthreads();
    const double part = (double)NRES / (double)sum[NTHREAD - 1];
    auto residue = [&](uint64_t before) { return min((uint32_t)((double)before * part), (uint32_t)NRES - 1u); };
    uint64_t at = upto - mine;
    for (int32_t k = k0; k < k1; k++) {
        const uint32_t c = cls[k];
        atomicAdd(&cnt[residue(at) * RANK_CLASSES + c], 1u);
        at += class_cost(c);
    }
    __syncthreads();
    /* exclusive prefix of each residue's class counts, heaviest class first */
    const uint32_t x8 = tid / RANK_CLASSES;
    if (counts) {
        const uint32_t c = RANK_CLASSES - 1u - tid % RANK_CLASSES;
        const uint32_t v = cnt[x8 * RANK_CLASSES + c], incl = wave_incl_scan(v);
        fill[x8 * RANK_CLASSES + c] = incl - v;
        if (c == 0) rtot[x8] = incl;
    }
    __syncthreads();
    /* unit of residue x at rank i goes to slot NRES * i + x */
    const uint32_t cap = (uint32_t)d.nslots / NRES;
    auto place = [&](int32_t k, uint32_t x, uint32_t pos) {
        if (pos >= cap) {                           /* the n-th unit without a slot */
            uint32_t n = pos - cap;
            for (uint32_t y = 0; y < x; y++) n += max(rtot[y], cap) - cap;
            for (x = 0; n >= cap - min(rtot[x], cap); x++) n -= cap - min(rtot[x], cap);
            pos = rtot[x] + n;
        }
        perm[NRES * pos + x] = k;
    };
    if (d.dmax <= RANK_ORDERED_DMAX || d.ntiles <= 512) {
        at = upto - mine;
        for (int32_t k = k0; k < k1; k++) {
            const uint32_t c = cls[k], x = residue(at);
            at += class_cost(c);
            place(k, x, atomicAdd(&fill[x * RANK_CLASSES + c], 1u));
        }
    } else if (counts) {
        /* a wavefront per run, 64 units at a time, so that the units of a class
         * keep their order */
        const uint32_t lane = tid & (WAVE - 1);
        int32_t b = 0;
        for (uint32_t y = 0; y < x8; y++) b += (int32_t)rtot[y];
        for (const int32_t end = b + (int32_t)rtot[x8]; b < end; b += WAVE) {
            const int32_t k = b + (int32_t)lane;
            const uint32_t c = k < end ? cls[k] : 0u;
            const uint64_t m = same_lanes<6>(c, ballot64(k < end));
            const uint32_t before = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            const uint32_t pos = fill[x8 * RANK_CLASSES + c] + before;
            wave_sync();
            if (k < end && before == 0u) fill[x8 * RANK_CLASSES + c] += (uint32_t)__popcll(m);
            wave_sync();
            if (k < end) place(k, x8, pos);
        }
    }
    /* the remaining slots are empty */
    uint32_t over = 0;
    for (uint32_t y = 0; y < NRES; y++) over += max(rtot[y], cap) - cap;
    for (int32_t i = tid; i < d.nslots; i += NTHREAD) {
        const uint32_t x = (uint32_t)i % NRES, pos = (uint32_t)i / NRES;
        if (pos < rtot[x]) continue;
        uint32_t n = pos - rtot[x];                 /* free slots before this one */
        for (uint32_t y = 0; y < x; y++) n += cap - min(rtot[y], cap);
        if (n >= over) perm[i] = -1;
    }
}

/* The kernel's first argument, read again from its segment: the compiler keeps
 * what it loads from here in registers only while it is used, and not, as the
 * argument's own fields, from the kernel's start to its end (some sixty pointers
 * and sizes: 77 to 82 scalar registers went to spills with units of 384; a sweep
 * of 96 chains 28.5 us per cycle so, 27.7 with this). */
__device__ __forceinline__ const bsim_dev &args_again()
{
    typedef const __attribute__((address_space(4))) char *kptr;
    kptr p = (kptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const bsim_dev *)p;
}

/* Phase (i) of cycle t: an owner thread updates its targets of unit id, with
 * the input that phase (ii) left in acc. */
template <int S_, bool PRE>
__device__ __forceinline__ void update_unit(int32_t id, int32_t t, uint32_t U, const Acc<S_> &acc,
                                            const NState<PRE ? S_ : 1> &ns)
{
    const uint32_t lane = threadIdx.x & (WAVE - 1), w = wave_index();
    const bsim_dev &d = args_again();
    const int32_t D = d.dmax;
    const uint64_t dmask = (D >= 63) ? (~0ull >> 1) : ((1ull << D) - 1ull);
    const int32_t base = id * (int32_t)U;
    const uint64_t *hist_in = d.hist + (int64_t)((t - 1) & 1) * d.n;
    uint64_t *hist_out = d.hist + (int64_t)(t & 1) * d.n;
    uint32_t *cnt_out = d.seg_count + (int64_t)(t & 1) * d.nwords;
    uint16_t *seg_out = d.seg + (int64_t)(t & 1) * d.nwords * (WAVE * D);
    const bool rec = d.raster != nullptr && t >= d.rec_t0 && t < d.rec_t0 + d.rec_steps;
#pragma unroll
    for (int j = 0; j < S_; j++) {
        const uint32_t i0 = (w - NEV) * WAVE + j * (NOWN * WAVE);
        if (i0 >= U) continue;                            /* uniform */
        const int32_t n0 = base + (int32_t)i0;
        const int32_t nid = n0 + (int32_t)lane;
        const bool valid = nid < d.n;
        bool fired = false;
        uint64_t h = 0;
        if (valid) {
            uint32_t cls;
            int32_t rs;
            float v, ie, ii, vtmp;
            uint64_t hin;
            if constexpr (PRE) {
                cls = ns.cls[j]; rs = ns.refrac[j]; v = ns.v[j]; ie = ns.ie[j]; ii = ns.ii[j];
                vtmp = ns.vtmp[j]; hin = ns.hist[j];
            } else {
                cls = d.ncls[nid]; rs = d.refrac[nid]; v = d.v[nid]; ie = d.ie[nid]; ii = d.ii[nid];
                vtmp = d.v_tmp[nid]; hin = hist_in[nid];
            }
            const uint32_t kind = cls >> 30;
            if (kind == BSIM_KIND_LIF) {
                const float inE = acc.e[j];
                const float inI = acc.i[j];
                if (rs > 0) {
                    d.refrac[nid] = rs - 1;
                } else {
                    bsim_lifc c;
                    if constexpr (PRE) c = ns.c[j]; else c = d.lifc[cls & BSIM_CLS_SET_MASK];
                    v = c.Cm * v + vtmp + ie * c.C_E + ii * c.C_I;
                    ie = c.CE * ie;
                    ii = c.CI * ii;
                    if (v >= c.v_thresh) {
                        fired = true;
                        d.refrac[nid] = c.refrac_time - 1;
                        v = c.v_reset;
                    } else {
                        if (d.in_sum) d.in_sum[nid] = d.in_sum[nid] + (inE + inI);
                        ie += inE;
                        ii += inI;
                    }
                    d.v[nid] = v;
                    d.ie[nid] = ie;
                    d.ii[nid] = ii;
                }
            } else if (kind == BSIM_KIND_ARRAY) {
                const int32_t c = d.arr_cur[nid];
                if (c < d.arr_end[nid] && d.arr_t[c] <= t) {
                    fired = true;
                    d.arr_cur[nid] = c + 1;
                }
            } else if (kind == BSIM_KIND_POISSON) {
                /* PoissonNeuron::update (src/neuron/poisson/PoissonNeuron.cpp:52-63):
                 * fire at the drawn cycle before the end cycle, then draw
                 * the next one 1 + X cycles later */
                const int32_t nx = d.arr_cur[nid];
                if (t == nx && nx < d.arr_end[nid]) {
                    fired = true;
                    const uint32_t x = poisson_pick(d.pois_tab + d.bern_p[nid],
                                                    bern_hash(d.bern_seed[nid], d.bern_key[nid], (uint32_t)t));
                    d.arr_cur[nid] = (int32_t)min((int64_t)nx + 1 + x, (int64_t)0x7FFFFFFF);
                }
            } else {
                fired = bern_hash(d.bern_seed[nid], d.bern_key[nid], (uint32_t)t) < d.bern_p[nid];
            }
            h = (hin << 1) | (fired ? 1ull : 0ull);
            hist_out[nid] = h;
            if (d.slot_count) d.slot_count[nid] += __popcll((h >> 1) & dmask);
            if (fired) d.fire_count[nid] += 1;
            if (rec && d.rec_index) {
                const int32_t ri = d.rec_index[nid];
                if (ri >= 0) {
                    const int64_t o = (int64_t)(t - d.rec_t0) * d.n_rec + ri;
                    d.rec_v[o] = kind == BSIM_KIND_LIF ? v : 0.0f;
                    if (d.rec_ie) {
                        d.rec_ie[o] = kind == BSIM_KIND_LIF ? ie : 0.0f;
                        d.rec_ii[o] = kind == BSIM_KIND_LIF ? ii : 0.0f;
                        d.rec_in_e[o] = kind == BSIM_KIND_LIF ? acc.e[j] : 0.0f;
                        d.rec_in_i[o] = kind == BSIM_KIND_LIF ? acc.i[j] : 0.0f;
                    }
                }
            }
        }
        const uint64_t fm = ballot64(fired);
        /* the block's list of active rows: each neuron's delays that
         * deliver in phase (ii) of this cycle, in order */
        uint64_t m = valid ? (h >> 1) & dmask : 0ull;
        const uint32_t c = (uint32_t)__popcll(m), incl = wave_incl_scan(c);
        if (n0 < d.n) {                                   /* uniform */
            uint16_t *out = seg_out + (int64_t)(n0 / 64) * (WAVE * D) + (incl - c);
            for (; m; m &= m - 1) *out++ = (uint16_t)(lane << 6 | (uint32_t)__builtin_ctzll(m));
            if (lane == WAVE - 1) cnt_out[n0 / 64] = incl;
            if (lane == 0 && rec) d.raster[(int64_t)(t - d.rec_t0) * d.nwords + n0 / 64] = fm;
        }
    }
}

/* The batch's rows, once every chunk has been summed; how many there are. */
__device__ __forceinline__ uint32_t batch_rows(const Shared &S, int32_t nrb, uint32_t buf, Rows &R)
{
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    R.nrb = nrb;
    R.at = 0;
    R.end = wave_incl_scan((int32_t)lane < nrb ? S.ctot[buf * MAXR + lane] : 0u);
    return readlane(R.end, WAVE - 1);
}

/* Event wavefronts: the unit of record k (below 0: none). */
template <int NB, int WR>
__device__ __forceinline__ void event_unit(const Shared &S, int32_t k, int32_t t, bool deliver, bool clocked,
                                           uint32_t U, uint32_t K, uint32_t &par, uint32_t &nb)
{
    const bsim_dev &d = args_again();
    const bsim_unit *un = d.unit + (k < 0 ? 0 : k);
    const int32_t id = k < 0 ? -1 : un->id, list = (t - 1) & 1;
    const int32_t nrng = deliver && id >= 0 ? un->nrng : 0;
    uint32_t events = 0, rows = 0;
    for (int32_t rb = 0; rb < nrng; rb += MAXR) {
        const int32_t nrb = min(MAXR, nrng - rb);
        prepare_batch(S, d, un, rb, nrb, list, nb);
        wg_barrier();
        Rows R;
        const uint32_t nrows = batch_rows(S, nrb, nb, R);
        nb ^= 1u;
        rows += nrows;
        if (nrows > 0)                          /* uniform */
            event_wave<NB, WR>(S, d, (uint32_t)un->part * U, un->nsyn, R, nrows,
                               d.seg + (int64_t)list * d.nwords * (WAVE * d.dmax), U, K, par, d.syn + un->base,
                               events);
    }
    /* the unit's work in this launch, when the next one ranks the units: its
     * deliveries plus a fixed cost of two deliveries per active row, x 16 */
    if (threadIdx.x == 0 && rows > 0) {
        atomicAdd((unsigned long long *)&d.ev_count[id], (unsigned long long)events);
        const int32_t re = d.rank_every;
        if (clocked && re > 0 && (t + 1) % re == 0)
            d.tile_load[(int64_t)(t & 1) * d.ntiles + id] = (uint64_t)events * 16ull + (uint64_t)rows * 32ull;
    }
}

/* Owner wavefronts: the same unit's sums and update. */
template <int S_>
__device__ __forceinline__ void owner_unit(const Shared &S, int32_t k, int32_t t, bool deliver, bool update,
                                           uint32_t U, uint32_t K, uint32_t &par, uint32_t &nb)
{
    constexpr bool PRE = S_ <= PREFETCH_MAX_S;
    const bsim_dev &d = args_again();
    const bsim_unit *un = d.unit + (k < 0 ? 0 : k);
    const int32_t id = k < 0 ? -1 : un->id;
    const int32_t nrng = deliver && id >= 0 ? un->nrng : 0;
    const bool upd = update && id >= 0;
    Acc<S_> acc;
#pragma unroll
    for (int j = 0; j < S_; j++) {
        acc.e[j] = 0.0f;
        acc.i[j] = 0.0f;
    }
    NState<PRE ? S_ : 1> ns;
    if constexpr (PRE) {
        if (upd) {
            load_nstate<S_>(d, id * (int32_t)U, d.hist + (int64_t)((t - 1) & 1) * d.n, ns);
            load_params<S_>(d, ns);
        }
    }
    for (int32_t rb = 0; rb < nrng; rb += MAXR) {
        wg_barrier();
        Rows R;
        const uint32_t nrows = batch_rows(S, min(MAXR, nrng - rb), nb, R);
        nb ^= 1u;
        if (nrows > 0) owner_wave<S_>(S, U, K, par, acc);     /* uniform */
    }
    if (upd) update_unit<S_, PRE>(id, t, U, acc, ns);
}

/* ONE: the grid's one unit, cycles cycles from the clock's on; otherwise one cycle. */
template <int NB, int WR, int S_, bool ONE>
__global__ __launch_bounds__(NTHREAD, STEP_EU) void bsim_step_kernel(bsim_dev d, int32_t t, int32_t flags,
                                                                     int32_t cycles)
{
    extern __shared__ __align__(16) uint32_t lds[];
    const bool clocked = t < 0;
    if (clocked) {
        t = device_cycle(d, blockIdx.x % 8u);
        flags = (t > 0 ? 1 : 0) | 2;
    }
    const int32_t re = d.rank_every;
    if ((int32_t)blockIdx.x < d.rank_wgs) {
        if (clocked) {
            /* orders the units for the launches from the next one on, by the
             * work that the launch before recorded */
            if (blockIdx.x == 0 && re > 0 && t > 0 && t % re == 0)
                rank_units(d, d.tile_load + (int64_t)((t - 1) & 1) * d.ntiles,
                           d.perm + (int64_t)((t / re) & 1) * d.nslots, lds, (uint32_t)lds_bytes((uint32_t)d.tile));
            wg_barrier();
            if (threadIdx.x == 0) count_done(d, 1u);
        }
        return;
    }
    const uint32_t U = (uint32_t)d.tile, K = slots_of(U);
    /* the workgroup's unit record: the slot's own, or in the order of the last ranking */
    int32_t k = (int32_t)blockIdx.x - d.rank_wgs;
    if (d.rank_wgs > 0) k = d.perm[(re > 0 && t > 0 ? (int64_t)(((t - 1) / re) & 1) * d.nslots : 0) + k];
    const uint32_t tid = threadIdx.x, w = wave_index();

    Shared S;
    {
        S.chunk = reinterpret_cast<Chunk *>(lds);
        S.hist = reinterpret_cast<uint32_t *>(S.chunk + MAXR);
        S.mark = S.hist + 2 * U * (NCOL / 4);
        S.slot = reinterpret_cast<float *>(S.mark + 2 * PASS);
        S.blk_end = reinterpret_cast<uint32_t *>(S.slot + K * U);
        S.blk_mark = S.blk_end + MAXR * BLKS;
        S.btot = S.blk_mark + NEV * WAVE;
        S.ctot = S.btot + 2 * NEV;
        S.most = S.ctot + 2 * MAXR;
        S.last = S.most + 2;
    }

    const bool deliver = (flags & 1) != 0, update = (flags & 2) != 0;
    if (deliver || ONE) {
        for (uint32_t i = tid; i < 2 * U; i += NTHREAD)
            reinterpret_cast<uint4 *>(S.hist)[i] = make_uint4(0u, 0u, 0u, 0u);
        for (uint32_t i = tid; i < 2 * PASS; i += NTHREAD) S.mark[i] = NO_MARK;
        if (w < NEV) S.blk_mark[tid] = NO_MARK;
        if (tid < 4) S.most[tid] = 0u;          /* most and last */
    }
    uint32_t par = 0, nb = 0;       /* passes and batches so far, modulo 2 */
    if (ONE && clocked) {
        /* what the owner wavefronts write in a cycle, this workgroup's event
         * wavefronts read in the next: a barrier in between orders that */
        if (w < NEV) {
            for (int32_t c = 0; c < cycles; c++, t++) {
                event_unit<NB, WR>(S, k, t, t > 0, true, U, K, par, nb);
                wg_barrier();
            }
        } else {
            for (int32_t c = 0; c < cycles; c++, t++) {
                owner_unit<S_>(S, k, t, t > 0, true, U, K, par, nb);
                wg_barrier();
            }
        }
        if (tid == 0) count_done(d, (uint64_t)cycles);
        return;
    }
    if (w < NEV)
        event_unit<NB, WR>(S, k, t, deliver, clocked, U, K, par, nb);
    else
        owner_unit<S_>(S, k, t, deliver, update, U, K, par, nb);
    if (clocked) wg_barrier();      /* every wavefront has read the cycle */
    if (clocked && tid == 0) count_done(d, 1u);
}

#ifdef STEP_MANY
extern "C" hipError_t bsim_launch_step_many(const bsim_dev *d, int32_t t, int32_t flags, hipStream_t stream)
{
    const uint32_t U = (uint32_t)d->tile;
    if (U == 0 || U % WAVE != 0 || U > NOWN * WAVE) return hipErrorInvalidValue;
    const dim3 grid(d->nslots + d->rank_wgs), block(NTHREAD);
    const size_t lds = lds_bytes(U);
    (void)hipGetLastError();       /* the check below then reports this launch alone */
#define STEP(NB) hipLaunchKernelGGL((bsim_step_kernel<NB, 1, 1, false>), grid, block, lds, stream, *d, t, flags, 1)
    if (U <= 64) STEP(6);
    else if (U <= 128) STEP(7);
    else STEP(8);
#undef STEP
    return hipGetLastError();
}
#else
extern "C" hipError_t bsim_launch_step_many(const bsim_dev *d, int32_t t, int32_t flags, hipStream_t stream);

/* One cycle, or with one unit (d.nslots 8, the others empty) and clocked as many
 * as cycles says: the launch and what a workgroup reads at its start are over
 * half of a small network's cycle.  us per cycle in runs, a launch each / 64 cycles a
 * launch: 48 neurons 5.1 / 3.0, 180 4.6 / 2.8, 250 with delays up to 30 steps 6.3
 * / 4.1. */
extern "C" hipError_t bsim_launch_step(const bsim_dev *d, int32_t t, int32_t flags, int32_t cycles,
                                       hipStream_t stream)
{
    if (d->ntiles <= 0) return hipSuccess;
    const uint32_t U = (uint32_t)d->tile;
    if (U == 0 || U % WAVE != 0 || U > BSIM_MAX_UNIT) return hipErrorInvalidValue;
    if (cycles != 1 && (t >= 0 || d->ntiles != 1)) return hipErrorInvalidValue;
    if (d->many) return bsim_launch_step_many(d, t, flags, stream);
    const dim3 grid(d->nslots + d->rank_wgs), block(NTHREAD);
    const size_t lds = lds_bytes(U);
    (void)hipGetLastError();       /* the check below then reports this launch alone */
#define OWN(X) (((X) + NOWN * WAVE - 1) / (NOWN * WAVE))
#define LAUNCH(NB, WR, X, ONE) \
    hipLaunchKernelGGL((bsim_step_kernel<NB, WR, OWN(X), ONE>), grid, block, lds, stream, *d, t, flags, cycles)
#define STEP(NB, X)                                    \
    do {                                               \
        if (d->ntiles == 1) LAUNCH(NB, 1, X, true);    \
        else if (d->wrows == 2) LAUNCH(NB, 2, X, false); \
        else LAUNCH(NB, 1, X, false);                  \
    } while (0)
    if (U <= 64) STEP(6, 64);
    else if (U <= 128) STEP(7, 128);
    else if (U <= 256) STEP(8, 256);
    else STEP(9, 512);
#undef OWN
#undef LAUNCH
#undef STEP
    return hipGetLastError();
}
#endif
