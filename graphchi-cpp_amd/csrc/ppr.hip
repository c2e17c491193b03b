// Batched personalized PageRank: many restart sets swept together.
//
// Kernel per query (the functional kernel with a seed-set restart, see
// example_apps/pagerank_functional.cpp:72-75 for the apply form):
//   r_v = (v in S ? (1 - d)/|S| : 0) + d * sum_{u -> v} r_u / outdeg_u
// iterated from r = teleport vector.  Every term is non-negative, so the
// iterates increase monotonically to the fixed point r*, and with
// res_k = ||r_k - r_{k-1}||_1 the remaining error is at most
// res_k * d / (1 - d); a query is converged when that bound is <= tol.
//
// Layout: 64 queries form a block; ranks are stored row-major, 64 values per
// vertex (128 B in BF16, 256 B in FP32), so every in-edge is one coalesced row
// gather shared by the 64 queries and the in-edge stream is read once per query
// block instead of once per query.  A last block of at most 32 queries has rows
// of 4, 8, 16 or 32 values.  Vertices with in-edges come first, in id order,
// then the others: a row without in-edges keeps its teleport value, written once.
//
// Work: the batch keeps the in-edges as one stream in row order (source
// position, 1/outdeg), a bit per edge that ends its row, and cuts it into items
// of S edges.  Every item is the same work whatever the row lengths are: a
// wavefront walks an item's edges with 16 gathers in flight and 16 more behind
// them, across row ends, and writes the rows that lie inside; the rows that
// cross items are summed from their parts by ppr_split_kernel.  (The form
// before took rows of up to 2W edges one at a time, a chain of five dependent
// loads each, from tiles too coarse to fill the chip with a small graph.)
// Bound: L2 and Infinity Cache reads of the rows in FP32, the wavefronts' issue
// rate in BF16.  R-MAT scale 17, 2.1M edges, 130 queries (64 + 64 + 2), one
// sweep: FP32 559 -> 107 us (1.07 GB of rows, 10 TB/s), BF16 501 -> 97 us, and
// 14 for the rows that cross items.  A sweep with the residuals, the last of every
// chunk, takes 150 and 32 in either precision.
//
// Precision: phase 1 stores ranks in BF16 with FP32 accumulation; phase 2
// converts to FP32 and refines with FP32 sweeps until every query meets the
// tolerance.  The per-query L1 residuals are FP64 sums.
#include "common.hpp"
#include "internal.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace gchi {
// plan internals shared with pagerank.hip
struct PlanView {
    uint32_t N, nhub, nchunk;
    uint64_t nedges;
    const uint32_t *reg_off, *reg_src, *hub_bits, *hub_v, *hub_chunk_off;
    const uint64_t *chunk_beg;
    const uint32_t *chunk_len, *hub_src, *outdeg;
};
int pr_plan_view(const gchi_pr_plan *p, PlanView *v);

// Kernel arguments: the batch's stream and tables.
struct PpArgs {
    const uint32_t *src;       // [E, padded] position of each edge's source
    const float *w;            // [E, padded] 1 / outdeg of the source (0 in the padding)
    const uint64_t *ends;      // bit e: edge e is the last of its row
    const uint32_t *item;      // [nitems] row of the item's first edge, | kPpMid when it began before
    const uint32_t *split;     // [nitems] row that begins in the item and goes on in the next; kPpNone
    const uint32_t *rstart;    // [K + 1] first edge of row k
    const uint32_t *pos, *vert;  // vertex -> position, position -> vertex
    const uint32_t *seedk;     // [nqb][kwords] bit k: row k is a seed of the block
    const uint32_t *seed_v, *seed_q, *seed_n;
    const float *tele;
    float *part;               // [nqb][nitems][2][64] head and tail sums of the rows that cross items
    double *res;
    const uint32_t *active;    // query blocks still swept; active[nqb] = their count
    uint32_t N, K, S, nitems, kwords, nqb;
    int lq;                    // the last block's rows have 2^lq values (6: like the others)
    uint64_t E;
    float damping;
};
}  // namespace gchi

struct gchi_ppr_batch {
    gchi::PpArgs a{};
    uint32_t nq = 0, nqb = 0, N = 0;
    size_t state = 0;              // values of one state buffer: [N][64] per query block, [N][2^lq] for the last
    void *r16[2] = {nullptr, nullptr};   // bf16
    float *r32[2] = {nullptr, nullptr};  // fp32
    double *res = nullptr;         // [nqb*64]
    uint32_t *seedk = nullptr;
    uint32_t *seed_v = nullptr;    // [nqb][64*64] sorted (vertex, query)
    uint32_t *seed_q = nullptr;
    uint32_t *seed_n = nullptr;    // [nqb]
    float *tele = nullptr;         // [nqb*64] restart mass per seed
    uint32_t *active = nullptr;    // [nqb] query blocks still swept, then their count at [nqb]
    int cur = 0;                   // buffer holding the current ranks
    int ncu = 256;
    bool fp32 = false;
    void *mem = nullptr;
    // chunks of sweeps captured once per phase and replayed (the residual is
    // read back only after each chunk)
    hipGraphExec_t chunk_exec[2] = {nullptr, nullptr};  // [0] BF16, [1] FP32
    hipGraph_t chunk_graph[2] = {nullptr, nullptr};
    int chunk_len[2] = {0, 0};
    float chunk_damping[2] = {0.0f, 0.0f};
};

namespace gchi {

constexpr int kPpThreads = 256;
constexpr int kPpWaves = kPpThreads / kWave;
constexpr int kQ = 64;                 // queries per block (one per lane)
constexpr int kMaxSeeds = 64;          // restart-set size limit per query
constexpr int kSeedTable = kQ * kMaxSeeds;
constexpr uint32_t kPpMid = 0x80000000u;
constexpr uint32_t kPpNone = 0xffffffffu;

GCHI_DEV float bf16_to_f32(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
GCHI_DEV uint16_t f32_to_bf16(float f) {  // round to nearest even
    uint32_t u = __float_as_uint(f);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}

template <typename T>
struct Store;
template <>
struct Store<uint16_t> {
    static GCHI_DEV float ld(const uint16_t *p) { return bf16_to_f32(*p); }
    static GCHI_DEV float round(float f) { return bf16_to_f32(f32_to_bf16(f)); }
    static GCHI_DEV void st(uint16_t *p, float f) { *p = f32_to_bf16(f); }
};
template <>
struct Store<float> {
    static GCHI_DEV float ld(const float *p) { return *p; }
    static GCHI_DEV float round(float f) { return f; }
    static GCHI_DEV void st(float *p, float f) { *p = f; }
};

// log2 of the values per row of query block qb; offset of its state
GCHI_DEV int pp_lq(const PpArgs &a, uint32_t qb) { return qb + 1 == a.nqb ? a.lq : 6; }
GCHI_DEV size_t pp_base(const PpArgs &a, uint32_t qb) { return (size_t)qb * a.N * kQ; }

// restart mass of (vertex v, query q of block qb), v known to be a seed of the block
GCHI_DEV float seed_mass(const PpArgs &a, uint32_t qb, uint32_t v, uint32_t q) {
    const uint32_t *sv = a.seed_v + (size_t)qb * kSeedTable;
    const uint32_t *sq = a.seed_q + (size_t)qb * kSeedTable;
    uint32_t lo = 0, hi = a.seed_n[qb];
    while (lo < hi) {
        uint32_t mid = (lo + hi) >> 1;
        if (sv[mid] < v) lo = mid + 1;
        else hi = mid;
    }
    float m = 0.0f;
    for (uint32_t k = lo; k < a.seed_n[qb] && sv[k] == v; k++)
        if (sq[k] == q) m = a.tele[qb * kQ + q];
    return m;
}

GCHI_DEV bool is_seed(const PpArgs &a, uint32_t qb, uint32_t k) {
    return (a.seedk[(size_t)qb * a.kwords + (k >> 5)] >> (k & 31)) & 1u;
}

GCHI_DEV float lane_f(float v, uint32_t l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), (int)l));
}

// What a wavefront knows of its item while it walks it (wavefront-uniform).
struct PpWalk {
    uint32_t k;       // row in progress
    bool mid;         // it began before the item
    uint32_t sw;      // seed bits of the rows 32 * (k / 32) ..
};

// The 64-edge groups of an item: source positions and weights of one group in
// lanes, the next group's loads in flight behind it.
struct PpGroup {
    uint32_t my, ny;
    float mw, nw;
    uint64_t f, nf;   // row ends
};

GCHI_DEV void pp_groups_open(const PpArgs &a, uint64_t e0, PpGroup &g, int lane) {
    g.my = __builtin_nontemporal_load(a.src + e0 + lane);
    g.mw = __builtin_nontemporal_load(a.w + e0 + lane);
    g.ny = __builtin_nontemporal_load(a.src + e0 + kWave + lane);  // padded past E
    g.nw = __builtin_nontemporal_load(a.w + e0 + kWave + lane);
    g.f = a.ends[e0 >> 6];
    g.nf = a.ends[(e0 >> 6) + 1];
}

// e: first edge of the new current group
GCHI_DEV void pp_groups_next(const PpArgs &a, uint64_t e, PpGroup &g, int lane) {
    g.my = g.ny;
    g.mw = g.nw;
    g.f = g.nf;
    g.ny = __builtin_nontemporal_load(a.src + e + kWave + lane);
    g.nw = __builtin_nontemporal_load(a.w + e + kWave + lane);
    g.nf = a.ends[(e >> 6) + 1];
}

// One item of 64 queries: lane = query, one row per load, two sets of 16 in
// flight.  (BF16 rows, two per load with half a wavefront each, took 174 us where
// this form took 141 with the same launch: the selects and shuffles cost more
// than the loads they save.  Sets of 4 / 8 / 16: 133 / 110 / 107 us in FP32.)
template <typename T, bool RES>
GCHI_DEV void pp_item(const PpArgs &a, uint32_t qb, uint32_t i, const T *__restrict__ Rin, T *__restrict__ Rout,
                      int lane, double *res) {
    constexpr uint32_t kSet = 16, kPerGroup = kWave / kSet;
    struct Set {
        float v[kSet], w[kSet];  // w is wavefront-uniform
        uint32_t f;
    };
    const uint64_t e0 = (uint64_t)i * a.S;
    const uint32_t n = (uint32_t)min<uint64_t>(a.S, a.E - e0), nb = (n + kSet - 1) / kSet;
    const uint32_t *sk = a.seedk + (size_t)qb * a.kwords;
    float *part = a.part + ((size_t)qb * a.nitems + i) * 2 * kQ + lane;
    PpGroup g;
    pp_groups_open(a, e0, g, lane);
    PpWalk k{a.item[i] & ~kPpMid, (a.item[i] & kPpMid) != 0, 0u};
    k.sw = sk[k.k >> 5];
    auto load = [&](Set &s, uint32_t b) {
        if (b >= nb) return;
        if (b && b % kPerGroup == 0) pp_groups_next(a, e0 + (uint64_t)kSet * b, g, lane);
        const uint32_t j = b % kPerGroup * kSet;
        s.f = (uint32_t)(g.f >> j) & ((1u << kSet) - 1u);
#pragma unroll
        for (uint32_t q = 0; q < kSet; q++) {
            const uint32_t id = (uint32_t)__builtin_amdgcn_readlane((int)g.my, (int)(j + q));
            s.w[q] = lane_f(g.mw, j + q);
            s.v[q] = Store<T>::ld(Rin + (size_t)id * kQ + lane);
        }
    };
    float acc = 0.0f, rn = 0.0f, ro = 0.0f;  // rn, ro: the row before, its residual not yet added
    auto end_row = [&]() {
        if (k.mid) {
            part[0] = acc;
            k.mid = false;
        } else {
            float m = 0.0f;
            if ((k.sw >> (k.k & 31)) & 1u) m = seed_mass(a, qb, a.vert[k.k], (uint32_t)lane);
            if (RES) *res += fabs((double)rn - (double)ro);
            rn = Store<T>::round(m + a.damping * acc);
            if (RES) ro = Store<T>::ld(Rin + (size_t)k.k * kQ + lane);
            Store<T>::st(Rout + (size_t)k.k * kQ + lane, rn);
        }
        acc = 0.0f;
        k.k++;
        if ((k.k & 31) == 0) k.sw = sk[k.k >> 5];
    };
    auto count = [&](const Set &s) {
        if (s.f == 0) {
#pragma unroll
            for (uint32_t q = 0; q < kSet; q++) acc += s.v[q] * s.w[q];
        } else {
#pragma unroll
            for (uint32_t q = 0; q < kSet; q++) {
                acc += s.v[q] * s.w[q];
                if ((s.f >> q) & 1u) end_row();
            }
        }
    };
    Set sa, sb;
    load(sa, 0);
    for (uint32_t b = 0;; b += 2) {
        load(sb, b + 1);
        count(sa);
        if (b + 1 >= nb) break;
        load(sa, b + 2);
        count(sb);
        if (b + 2 >= nb) break;
    }
    if (RES) *res += fabs((double)rn - (double)ro);
    // the row in progress: its first edge lies in this item (tail) or before (head)
    const uint64_t last = e0 + n - 1;
    if (!((a.ends[last >> 6] >> (last & 63)) & 1u)) part[k.mid ? 0 : kQ] = acc;
}

// 64 >> lq items, one per group of 2^lq lanes, for a last block of few queries.
// Each group walks its own item, 8 edges at a time.
template <typename T, bool RES>
GCHI_DEV void pp_items_narrow(const PpArgs &a, uint32_t qb, uint32_t first, const T *__restrict__ Rin,
                              T *__restrict__ Rout, int lane, double *res) {
    const int lq = a.lq;
    const uint32_t q = (uint32_t)lane & ((1u << lq) - 1u), i = first + ((uint32_t)lane >> lq);
    const bool on = i < a.nitems;
    const uint64_t e0 = on ? (uint64_t)i * a.S : 0ull;
    const uint32_t n = on ? (uint32_t)min<uint64_t>(a.S, a.E - e0) : 0u;
    float *part = a.part + ((size_t)qb * a.nitems + (on ? i : 0u)) * 2 * kQ + q;
    const uint32_t meta = on ? a.item[i] : 0u;
    uint32_t k = meta & ~kPpMid;
    bool mid = (meta & kPpMid) != 0;
    const uint8_t *ends = reinterpret_cast<const uint8_t *>(a.ends) + e0 / 8;
    float acc = 0.0f;
    for (uint32_t j = 0; j < n; j += 8) {
        const uint4 i0 = *reinterpret_cast<const uint4 *>(a.src + e0 + j);
        const uint4 i1 = *reinterpret_cast<const uint4 *>(a.src + e0 + j + 4);
        const float4 w0 = *reinterpret_cast<const float4 *>(a.w + e0 + j);
        const float4 w1 = *reinterpret_cast<const float4 *>(a.w + e0 + j + 4);
        const uint32_t id[8] = {i0.x, i0.y, i0.z, i0.w, i1.x, i1.y, i1.z, i1.w};
        const float w[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
        const uint32_t f = ends[j / 8];
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = Store<T>::ld(Rin + ((size_t)id[u] << lq) + q);
#pragma unroll
        for (int u = 0; u < 8; u++) {
            acc += v[u] * w[u];
            if ((f >> u) & 1u) {
                if (mid) {
                    part[0] = acc;
                    mid = false;
                } else {
                    float m = 0.0f;
                    if (is_seed(a, qb, k)) m = seed_mass(a, qb, a.vert[k], q);
                    const float rn = Store<T>::round(m + a.damping * acc);
                    const size_t at = ((size_t)k << lq) + q;
                    if (RES) *res += fabs((double)rn - (double)Store<T>::ld(Rin + at));
                    Store<T>::st(Rout + at, rn);
                }
                acc = 0.0f;
                k++;
            }
        }
    }
    if (on) {
        const uint64_t last = e0 + n - 1;
        if (!((a.ends[last >> 6] >> (last & 63)) & 1u)) part[mid ? 0 : kQ] = acc;
    }
}

// The units of a sweep: the narrow block's first (its chains are the longest),
// then kPpWaves items of one query block each, block by block.
struct PpUnits {
    uint32_t narrow, wide, total;  // units of the narrow block; of every wide one; of all
};

GCHI_DEV PpUnits pp_units(const PpArgs &a, uint32_t per_wave_wide, uint32_t items) {
    const uint32_t nact = a.active[a.nqb];
    const bool nar = a.lq < 6 && nact && a.active[nact - 1] == a.nqb - 1;
    PpUnits u;
    const uint32_t group = per_wave_wide * kPpWaves;
    u.wide = (items + group - 1) / group;
    u.narrow = nar ? (items + (group << (6 - a.lq)) - 1) / (group << (6 - a.lq)) : 0u;
    u.total = u.narrow + (nact - (nar ? 1u : 0u)) * u.wide;
    return u;
}

// Adds the workgroup's residuals of block qb to the global ones.
GCHI_DEV void pp_flush_res(const PpArgs &a, uint32_t qb, double *s_res) {
    __syncthreads();
    if (threadIdx.x < kQ) {
        const double v = s_res[threadIdx.x];
        if (v != 0.0) atomicAdd(&a.res[qb * kQ + threadIdx.x], v);
        s_res[threadIdx.x] = 0.0;
    }
    __syncthreads();
}

template <typename T, bool RES>
__global__ __launch_bounds__(kPpThreads) void ppr_sweep_kernel(PpArgs a, const T *__restrict__ Rin_all,
                                                              T *__restrict__ Rout_all) {
    __shared__ double s_res[kQ];
    const int lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const PpUnits un = pp_units(a, 1, a.nitems);
    uint32_t cur = kPpNone;
    if (RES) {
        if (threadIdx.x < kQ) s_res[threadIdx.x] = 0.0;
        __syncthreads();
    }
    for (uint32_t u = blockIdx.x; u < un.total; u += gridDim.x) {
        const bool nar = u < un.narrow;
        const uint32_t t = u - un.narrow, qi = nar ? 0u : t / un.wide;
        const uint32_t qb = nar ? a.nqb - 1 : a.active[qi];
        if (RES && qb != cur && cur != kPpNone) pp_flush_res(a, cur, s_res);  // block-uniform
        cur = qb;
        const T *Rin = Rin_all + pp_base(a, qb);
        T *Rout = Rout_all + pp_base(a, qb);
        double res = 0.0;
        if (nar) {
            pp_items_narrow<T, RES>(a, qb, (u * kPpWaves + wave) << (6 - a.lq), Rin, Rout, lane, &res);
            if (RES) atomicAdd(&s_res[lane & ((1 << a.lq) - 1)], res);
        } else {
            const uint32_t i = (t - qi * un.wide) * kPpWaves + wave;
            if (i < a.nitems) pp_item<T, RES>(a, qb, i, Rin, Rout, lane, &res);
            if (RES) atomicAdd(&s_res[lane], res);
        }
    }
    if (RES && cur != kPpNone) pp_flush_res(a, cur, s_res);
}

// The rows that cross items: the first item's tail, then the heads of the items
// after it up to the row's last, added in that order, 16 loads in flight.
template <typename T, bool RES>
__global__ __launch_bounds__(kPpThreads) void ppr_split_kernel(PpArgs a, const T *__restrict__ Rin_all,
                                                              T *__restrict__ Rout_all) {
    __shared__ double s_res[kQ];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    constexpr uint32_t kPer = 4;  // items per wavefront (or group) and unit: about half have such a row
    const PpUnits un = pp_units(a, kPer, a.nitems);
    uint32_t cur = kPpNone;
    if (RES) {
        if (threadIdx.x < kQ) s_res[threadIdx.x] = 0.0;
        __syncthreads();
    }
    for (uint32_t u = blockIdx.x; u < un.total; u += gridDim.x) {
        const bool nar = u < un.narrow;
        const uint32_t t = u - un.narrow, qi = nar ? 0u : t / un.wide;
        const uint32_t qb = nar ? a.nqb - 1 : a.active[qi];
        if (RES && qb != cur && cur != kPpNone) pp_flush_res(a, cur, s_res);
        cur = qb;
        const int lq = nar ? a.lq : 6;
        const uint32_t q = (uint32_t)lane & ((1u << lq) - 1u), groups = 64u >> lq;
        const T *Rin = Rin_all + pp_base(a, qb);
        T *Rout = Rout_all + pp_base(a, qb);
        const float *part = a.part + (size_t)qb * a.nitems * 2 * kQ + q;
        const uint32_t unit = nar ? u : t - qi * un.wide;
        const uint32_t i0 = ((unit * kPpWaves + wave) * groups + ((uint32_t)lane >> lq)) * kPer;
        double res = 0.0;
        for (uint32_t i = i0; i < min(i0 + kPer, a.nitems); i++) {
            const uint32_t k = a.split[i];
            if (k == kPpNone) continue;
            const uint32_t il = (a.rstart[k + 1] - 1) / a.S;
            float acc = part[(size_t)i * 2 * kQ + kQ];
            for (uint32_t c = i + 1; c <= il; c += 16) {
                float pv[16];
#pragma unroll
                for (uint32_t x = 0; x < 16; x++) pv[x] = part[(size_t)min(c + x, il) * 2 * kQ];
#pragma unroll
                for (uint32_t x = 0; x < 16; x++)
                    if (c + x <= il) acc += pv[x];
            }
            float m = 0.0f;
            if (is_seed(a, qb, k)) m = seed_mass(a, qb, a.vert[k], q);
            const float rn = Store<T>::round(m + a.damping * acc);
            const size_t at = ((size_t)k << lq) + q;
            if (RES) res += fabs((double)rn - (double)Store<T>::ld(Rin + at));
            Store<T>::st(Rout + at, rn);
        }
        if (RES && res != 0.0) atomicAdd(&s_res[q], res);
    }
    if (RES && cur != kPpNone) pp_flush_res(a, cur, s_res);
}

// ---- start values ----
// r = teleport vector: R0 cleared (all rows, or only those without in-edges),
// R1's rows without in-edges cleared; ppr_seed_kernel then writes the seeds.
template <typename T>
__global__ void ppr_clear_kernel(PpArgs a, T *__restrict__ R0, T *__restrict__ R1, int whole) {
    struct __align__(4 * sizeof(T)) Four {
        T x[4];
    };
    const Four zero = {};
    for (uint32_t qb = blockIdx.y; qb < a.nqb; qb += gridDim.y) {
        const int lq = pp_lq(a, qb);
        const size_t n4 = ((size_t)a.N << lq) / 4, k4 = ((size_t)a.K << lq) / 4;  // rows of at least 4 values
        Four *r0 = reinterpret_cast<Four *>(R0 + pp_base(a, qb)), *r1 = reinterpret_cast<Four *>(R1 + pp_base(a, qb));
        const size_t stride = (size_t)gridDim.x * blockDim.x;
        for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x + (whole ? 0 : k4); i < n4; i += stride) {
            r0[i] = zero;
            if (i >= k4) r1[i] = zero;
        }
    }
}

// The seeds' masses: rows without in-edges in both buffers, the others in R0
// (whole) with their bit in seedk.
template <typename T>
__global__ void ppr_seed_kernel(PpArgs a, T *__restrict__ R0, T *__restrict__ R1, uint32_t *seedk, int whole) {
    for (uint32_t qb = blockIdx.x; qb < a.nqb; qb += gridDim.x) {
        const int lq = pp_lq(a, qb);
        for (uint32_t e = threadIdx.x; e < a.seed_n[qb]; e += blockDim.x) {
            const uint32_t p = a.pos[a.seed_v[(size_t)qb * kSeedTable + e]];
            const uint32_t q = a.seed_q[(size_t)qb * kSeedTable + e];
            const size_t at = pp_base(a, qb) + ((size_t)p << lq) + q;
            const float m = a.tele[qb * kQ + q];
            if (whole || p >= a.K) Store<T>::st(R0 + at, m);
            if (p >= a.K) Store<T>::st(R1 + at, m);
            else atomicOr(&seedk[(size_t)qb * a.kwords + (p >> 5)], 1u << (p & 31));
        }
    }
}

__global__ void ppr_widen_kernel(const uint16_t *a, float *b, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) b[i] = bf16_to_f32(a[i]);
}

__global__ void ppr_extract_kernel(PpArgs a, const void *R, int fp32, uint32_t query, float *out) {
    uint32_t stride = gridDim.x * blockDim.x;
    const uint32_t qb = query / kQ, q = query % kQ;
    const int lq = pp_lq(a, qb);
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < a.N; v += stride) {
        const size_t i = pp_base(a, qb) + ((size_t)a.pos[v] << lq) + q;
        out[v] = fp32 ? ((const float *)R)[i] : bf16_to_f32(((const uint16_t *)R)[i]);
    }
}

// ---- stream build (once per batch) ----
GCHI_DEV bool pb_is_hub(const PlanView &p, uint32_t v) { return (p.hub_bits[v >> 5] >> (v & 31)) & 1u; }

__global__ void pb_lengths(PlanView p, uint32_t *len, uint32_t *some) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < p.N; v += stride) {
        if (p.nhub && pb_is_hub(p, v)) continue;
        const uint32_t l = p.reg_off[v + 1] - p.reg_off[v];
        len[v] = l;
        some[v] = l != 0;
    }
}

__global__ void pb_hub_lengths(PlanView p, uint32_t *len, uint32_t *some) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t h = blockIdx.x * blockDim.x + threadIdx.x; h < p.nhub; h += stride) {
        const uint32_t c0 = p.hub_chunk_off[h], c1 = p.hub_chunk_off[h + 1];
        const uint32_t l = c1 > c0 ? (uint32_t)(p.chunk_beg[c1 - 1] + p.chunk_len[c1 - 1] - p.chunk_beg[c0]) : 0u;
        len[p.hub_v[h]] = l;
        some[p.hub_v[h]] = l != 0;
    }
}

// positions and row starts, and the row-end bits (cleared before)
__global__ void pb_rows(uint32_t n, const uint32_t *len, const uint32_t *ord, const uint32_t *start, uint32_t *pos,
                        uint32_t *vert, uint32_t *rstart, uint32_t *ends) {
    const uint32_t stride = gridDim.x * blockDim.x, K = ord[n];
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride) {
        const uint32_t l = len[v], p = l ? ord[v] : K + (v - ord[v]);
        pos[v] = p;
        vert[p] = v;
        if (l) {
            rstart[p] = start[v];
            const uint32_t e = start[v] + l - 1;
            atomicOr(&ends[e >> 5], 1u << (e & 31));
        }
        if (v == 0) rstart[K] = start[n];
    }
}

GCHI_DEV void pb_edge(const PlanView &p, const uint32_t *pos, uint32_t u, uint32_t e, uint32_t *src, float *w) {
    src[e] = pos[u];
    w[e] = p.outdeg[u] ? 1.0f / (float)p.outdeg[u] : 0.0f;
}

// 16 lanes per regular row
__global__ void pb_regular(PlanView p, const uint32_t *pos, const uint32_t *start, uint32_t *src, float *w) {
    const uint32_t l16 = threadIdx.x & 15u, stride = gridDim.x * blockDim.x / 16;
    for (uint32_t v = (blockIdx.x * blockDim.x + threadIdx.x) / 16; v < p.N; v += stride) {
        if (p.nhub && pb_is_hub(p, v)) continue;
        const uint32_t b = p.reg_off[v], l = p.reg_off[v + 1] - b, s = start[v];
        for (uint32_t k = l16; k < l; k += 16) pb_edge(p, pos, p.reg_src[b + k], s + k, src, w);
    }
}

// one wavefront per hub chunk
__global__ void pb_hubs(PlanView p, const uint32_t *pos, const uint32_t *start, uint32_t *src, float *w) {
    const uint32_t lane = threadIdx.x & (kWave - 1), stride = gridDim.x * blockDim.x / kWave;
    for (uint32_t c = (blockIdx.x * blockDim.x + threadIdx.x) / kWave; c < p.nchunk; c += stride) {
        uint32_t lo = 0, hi = p.nhub - 1;  // the chunk's hub: the last with hub_chunk_off[h] <= c
        while (lo < hi) {
            const uint32_t m = (lo + hi + 1) / 2;
            if (p.hub_chunk_off[m] <= c) lo = m;
            else hi = m - 1;
        }
        const uint64_t b = p.chunk_beg[c];
        const uint32_t s = start[p.hub_v[lo]] + (uint32_t)(b - p.chunk_beg[p.hub_chunk_off[lo]]);
        for (uint32_t k = lane; k < p.chunk_len[c]; k += kWave) pb_edge(p, pos, p.hub_src[b + k], s + k, src, w);
    }
}

__global__ void pb_items(const uint32_t *rstart, const uint32_t *K_, uint32_t S, uint32_t nitems, uint32_t *item,
                         uint32_t *split) {
    const uint32_t stride = gridDim.x * blockDim.x, K = *K_;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < nitems; i += stride) {
        uint32_t at[2];
        for (int s = 0; s < 2; s++) {  // the last row that begins at or before the item's first / last edge
            const uint64_t e = s ? min<uint64_t>((uint64_t)(i + 1) * S, rstart[K]) - 1 : (uint64_t)i * S;
            uint32_t lo = 0, hi = K - 1;
            while (lo < hi) {
                const uint32_t m = lo + (hi - lo + 1) / 2;
                if (rstart[m] <= e) lo = m;
                else hi = m - 1;
            }
            at[s] = lo;
        }
        item[i] = at[0] | ((uint64_t)rstart[at[0]] < (uint64_t)i * S ? kPpMid : 0u);
        const bool begins = (uint64_t)rstart[at[1]] >= (uint64_t)i * S;
        const bool goes_on = (uint64_t)rstart[at[1] + 1] > (uint64_t)(i + 1) * S;
        split[i] = begins && goes_on ? at[1] : kPpNone;
    }
}

static PpArgs make_args(const gchi_ppr_batch *b, float damping) {
    PpArgs a = b->a;
    a.damping = damping;
    return a;
}

template <typename T, bool RES>
static void ppr_launch(gchi_ppr_batch *b, const PpArgs &a, const T *rin, T *rout, hipStream_t s) {
    // more workgroups than fit at once: the hardware hands the later ones out as
    // the first end (8 per CU, each looping over its units, took 153 us in FP32, 16
    // 135, 32 110, one per unit 113)
    const uint64_t units = (uint64_t)b->nqb * div_up(a.nitems, kPpWaves);
    const unsigned grid = (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(units, (uint64_t)b->ncu * 32));
    const unsigned sgrid = (unsigned)std::max<uint64_t>(1, std::min<uint64_t>(div_up(units, 4), (uint64_t)b->ncu * 32));
    hipLaunchKernelGGL((ppr_sweep_kernel<T, RES>), dim3(grid), dim3(kPpThreads), 0, s, a, rin, rout);
    hipLaunchKernelGGL((ppr_split_kernel<T, RES>), dim3(sgrid), dim3(kPpThreads), 0, s, a, rin, rout);
}

template <typename T>
static int ppr_sweep(gchi_ppr_batch *b, const T *rin, T *rout, float damping, int residual, hipStream_t s) {
    const PpArgs a = make_args(b, damping);
    if (residual) launch_fill_u64(reinterpret_cast<uint64_t *>(b->res), 0ull, (size_t)b->nqb * kQ, s);
    if (residual) ppr_launch<T, true>(b, a, rin, rout, s);
    else ppr_launch<T, false>(b, a, rin, rout, s);
    GCHI_LAUNCH_CHECK();
    return GCHI_OK;
}

// Captures `len` sweeps of one phase (0: BF16, 1: FP32) from buffer 0, the
// last one with the residual, into a graph kept by the batch; recaptured only
// when the chunk length or the damping changes.  The kernels read the active
// list from device memory, so retiring blocks needs no recapture.
static int ppr_capture_chunk(gchi_ppr_batch *b, int phase, int len, float d) {
    if (b->chunk_exec[phase] && b->chunk_len[phase] == len && b->chunk_damping[phase] == d) return GCHI_OK;
    if (b->chunk_exec[phase]) (void)hipGraphExecDestroy(b->chunk_exec[phase]);
    if (b->chunk_graph[phase]) (void)hipGraphDestroy(b->chunk_graph[phase]);
    b->chunk_exec[phase] = nullptr;
    b->chunk_graph[phase] = nullptr;
    hipStream_t cs;
    GCHI_HIP(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
    int st = GCHI_OK;
    hipError_t e = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) st = hip_fail(e, "hipStreamBeginCapture", __FILE__, __LINE__);
    if (st == GCHI_OK) {
        int s1 = GCHI_OK;
        for (int k = 0; k < len && s1 == GCHI_OK; k++) {
            const int res = k == len - 1;
            if (phase == 0)
                s1 = ppr_sweep<uint16_t>(b, (const uint16_t *)b->r16[k & 1], (uint16_t *)b->r16[(k + 1) & 1], d, res,
                                         cs);
            else
                s1 = ppr_sweep<float>(b, b->r32[k & 1], b->r32[(k + 1) & 1], d, res, cs);
        }
        e = hipStreamEndCapture(cs, &b->chunk_graph[phase]);
        if (s1 != GCHI_OK) st = s1;
        else if (e != hipSuccess) st = hip_fail(e, "hipStreamEndCapture", __FILE__, __LINE__);
    }
    if (st == GCHI_OK) {
        e = hipGraphInstantiate(&b->chunk_exec[phase], b->chunk_graph[phase], nullptr, nullptr, 0);
        if (e != hipSuccess) st = hip_fail(e, "hipGraphInstantiate", __FILE__, __LINE__);
    }
    (void)hipStreamDestroy(cs);
    if (st != GCHI_OK) {
        if (b->chunk_graph[phase]) (void)hipGraphDestroy(b->chunk_graph[phase]);
        b->chunk_graph[phase] = nullptr;
        b->chunk_exec[phase] = nullptr;
        return st;
    }
    b->chunk_len[phase] = len;
    b->chunk_damping[phase] = d;
    return GCHI_OK;
}

}  // namespace gchi

using namespace gchi;

extern "C" int gchi_ppr_batch_create(const gchi_pr_plan *plan, uint32_t nqueries, gchi_ppr_batch **out) {
    GCHI_CHECK(plan && out && nqueries > 0, GCHI_ERR_INVALID, "ppr_batch_create: bad argument");
    PlanView pv;
    GCHI_TRY(pr_plan_view(plan, &pv));  // before the batch exists: a refused plan leaks nothing
    GCHI_CHECK(pv.N < kPpMid, GCHI_ERR_UNSUPPORTED, "ppr_batch_create: N must be < 2^31");
    gchi_ppr_batch *b = new gchi_ppr_batch();
    b->nq = nqueries;
    {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess)
            b->ncu = prop.multiProcessorCount;
    }
    const uint32_t N = pv.N, nqb = (nqueries + kQ - 1) / kQ;
    const uint64_t E = pv.nedges;
    b->nqb = nqb;
    b->N = N;
    PpArgs &a = b->a;
    a.N = N;
    a.nqb = nqb;
    a.E = E;
    // the last block's row: the power of two that holds its queries, at least 4 (8-byte rows in BF16)
    const uint32_t rest = nqueries - (nqb - 1) * kQ;
    a.lq = 2;
    while ((1u << a.lq) < rest) a.lq++;
    // edges per item: about four items per resident wavefront, so that the last
    // round of items is short, within [64, 512] (longer items have fewer rows
    // that cross them and amortise their first loads)
    const uint64_t slots = (uint64_t)b->ncu * 8 * kPpWaves * 4;
    const uint64_t lanes = E * ((uint64_t)(nqb - 1) * kQ + (1u << a.lq)) / kQ;
    a.S = (uint32_t)std::min<uint64_t>(512, std::max<uint64_t>(1, lanes / slots / 64) * 64);
    a.nitems = (uint32_t)div_up(E, a.S);
    a.kwords = N / 32 + 1;
    const size_t state = ((size_t)(nqb - 1) * kQ + ((size_t)1 << a.lq)) * N, epad = (size_t)E + 2 * a.S + 2 * kWave;
    b->state = state;
    auto lay = [&](auto &c, auto get) {
        get(0, c.template take<uint32_t>(epad));              // src
        get(1, c.template take<float>(epad));                 // w
        get(2, c.template take<uint64_t>(epad / 64 + 2));     // ends
        get(3, c.template take<uint32_t>(a.nitems + 1));      // item
        get(4, c.template take<uint32_t>(a.nitems + 1));      // split
        get(5, c.template take<uint32_t>((size_t)N + 1));     // rstart
        get(6, c.template take<uint32_t>(N));                 // pos
        get(7, c.template take<uint32_t>(N));                 // vert
        get(8, c.template take<uint32_t>((size_t)nqb * a.kwords));  // seedk
        get(9, c.template take<uint32_t>((size_t)nqb * kSeedTable));
        get(10, c.template take<uint32_t>((size_t)nqb * kSeedTable));
        get(11, c.template take<uint32_t>(nqb));
        get(12, c.template take<float>((size_t)nqb * kQ));    // tele
        get(13, c.template take<float>((size_t)nqb * a.nitems * 2 * kQ + 1));  // part
        get(14, c.template take<double>((size_t)nqb * kQ));   // res
        get(15, c.template take<uint32_t>((size_t)nqb + 1));  // active
        get(16, c.template take<uint16_t>(state));
        get(17, c.template take<uint16_t>(state));
        get(18, c.template take<float>(state));
        get(19, c.template take<float>(state));
    };
    auto lay_scratch = [&](auto &c, auto get) {  // of the build
        for (int k = 0; k < 4; k++) get(k, c.template take<uint32_t>((size_t)N + 1));  // len, some, ord, start
        get(4, c.template take<char>(scan_workspace((size_t)N + 1)));
    };
    SizerAdapter za, zs;
    lay(za, [](int, void *) {});
    lay_scratch(zs, [](int, void *) {});
    if (device_alloc(&b->mem, za.z.off) != hipSuccess) {
        delete b;
        return fail(GCHI_ERR_HIP, "ppr_batch_create: hipMalloc failed (state " + std::to_string(za.z.off) + " bytes)");
    }
    void *scratch = nullptr;
    if (hipError_t e = pool_alloc(&scratch, zs.z.off, 0)) {
        (void)hipFree(b->mem);
        delete b;
        return hip_fail(e, "ppr_batch_create: scratch", __FILE__, __LINE__);
    }
    void *m[20], *t[5];
    Carver c(b->mem, za.z.off), sc(scratch, zs.z.off);
    lay(c, [&](int k, void *q) { m[k] = q; });
    lay_scratch(sc, [&](int k, void *q) { t[k] = q; });
    auto u32 = [&](int k) { return static_cast<uint32_t *>(m[k]); };
    float *w = static_cast<float *>(m[1]);
    a.src = u32(0);
    a.w = w;
    a.ends = static_cast<uint64_t *>(m[2]);
    a.item = u32(3);
    a.split = u32(4);
    a.rstart = u32(5);
    a.pos = u32(6);
    a.vert = u32(7);
    a.seedk = b->seedk = u32(8);
    a.seed_v = b->seed_v = u32(9);
    a.seed_q = b->seed_q = u32(10);
    a.seed_n = b->seed_n = u32(11);
    a.tele = b->tele = static_cast<float *>(m[12]);
    a.part = static_cast<float *>(m[13]);
    a.res = b->res = static_cast<double *>(m[14]);
    a.active = b->active = u32(15);
    b->r16[0] = m[16];
    b->r16[1] = m[17];
    b->r32[0] = static_cast<float *>(m[18]);
    b->r32[1] = static_cast<float *>(m[19]);
    uint32_t *tmp[4];
    for (int k = 0; k < 4; k++) tmp[k] = static_cast<uint32_t *>(t[k]);
    uint32_t *len = tmp[0], *some = tmp[1], *ord = tmp[2], *start = tmp[3];
    const size_t swb = scan_workspace((size_t)N + 1);
    auto build = [&]() -> int {
        const dim3 gv(grid_for(N, 256, 65536)), blk(256);
        launch_fill_u32(u32(2), 0u, 2 * (epad / 64 + 2), 0);
        launch_fill_u32(u32(0) + E, 0u, epad - E, 0);
        launch_fill_u32(reinterpret_cast<uint32_t *>(w) + E, 0u, epad - E, 0);
        hipLaunchKernelGGL(pb_lengths, gv, blk, 0, 0, pv, len, some);
        if (pv.nhub) hipLaunchKernelGGL(pb_hub_lengths, dim3(grid_for(pv.nhub, 256, 65536)), blk, 0, 0, pv, len, some);
        GCHI_TRY(exclusive_scan_u32(some, ord, N, t[4], swb, 0));
        GCHI_TRY(exclusive_scan_u32(len, start, N, t[4], swb, 0));
        hipLaunchKernelGGL(pb_rows, gv, blk, 0, 0, N, len, ord, start, u32(6), u32(7), u32(5), u32(2));
        hipLaunchKernelGGL(pb_regular, dim3(grid_for((uint64_t)N * 16, 256, 65536)), blk, 0, 0, pv, u32(6), start,
                           u32(0), w);
        if (pv.nchunk)
            hipLaunchKernelGGL(pb_hubs, dim3(grid_for((uint64_t)pv.nchunk * kWave, 256, 65536)), blk, 0, 0, pv, u32(6),
                               start, u32(0), w);
        if (a.nitems)
            hipLaunchKernelGGL(pb_items, dim3(grid_for(a.nitems, 256, 65536)), blk, 0, 0, u32(5), ord + N, a.S,
                               a.nitems, u32(3), u32(4));
        GCHI_LAUNCH_CHECK();
        GCHI_HIP(hipMemcpyAsync(&a.K, ord + N, 4, hipMemcpyDeviceToHost, 0));
        GCHI_HIP(hipDeviceSynchronize());
        return GCHI_OK;
    };
    const int st = build();
    pool_free(scratch, hipStreamSynchronize(0));
    if (st != GCHI_OK) {
        (void)hipFree(b->mem);
        delete b;
        return st;
    }
    *out = b;
    return GCHI_OK;
}

extern "C" int gchi_ppr_batch_destroy(gchi_ppr_batch *b) {
    if (!b) return GCHI_OK;
    for (int k = 0; k < 2; k++) {
        if (b->chunk_exec[k]) (void)hipGraphExecDestroy(b->chunk_exec[k]);
        if (b->chunk_graph[k]) (void)hipGraphDestroy(b->chunk_graph[k]);
    }
    if (b->mem) (void)hipFree(b->mem);
    delete b;
    return GCHI_OK;
}

// Runs every query to convergence.  h_seed_off[nq+1] / h_seeds: restart sets.
extern "C" int gchi_ppr_batch_run(gchi_ppr_batch *b, const uint32_t *h_seed_off, const uint32_t *h_seeds,
                                  const gchi_ppr_config *cfg, gchi_ppr_result *result, double *h_residuals,
                                  void *stream) {
    GCHI_CHECK(b && h_seed_off && h_seeds && cfg && result, GCHI_ERR_INVALID, "ppr_batch_run: null argument");
    GCHI_CHECK(cfg->damping > 0 && cfg->damping < 1 && cfg->tol > 0, GCHI_ERR_INVALID, "ppr_batch_run: bad config");
    hipStream_t s = as_stream(stream);
    const uint32_t nqb = b->nqb, N = b->N;
    // seed tables (host-built, uploaded once per run)
    std::vector<uint32_t> sv((size_t)nqb * kSeedTable, 0), sq((size_t)nqb * kSeedTable, 0), sn(nqb, 0);
    std::vector<float> tele((size_t)nqb * kQ, 0.0f);
    for (uint32_t q = 0; q < b->nq; q++) {
        uint32_t k0 = h_seed_off[q], k1 = h_seed_off[q + 1];
        GCHI_CHECK(k1 > k0 && k1 - k0 <= (uint32_t)kMaxSeeds, GCHI_ERR_UNSUPPORTED,
                   "ppr_batch_run: each query needs 1..64 seeds");
        std::vector<uint32_t> seeds(h_seeds + k0, h_seeds + k1);
        std::sort(seeds.begin(), seeds.end());
        GCHI_CHECK(std::adjacent_find(seeds.begin(), seeds.end()) == seeds.end(), GCHI_ERR_INVALID,
                   "ppr_batch_run: repeated seed in a restart set");
        const uint32_t qb = q / kQ, lane = q % kQ;
        tele[q] = (float)((1.0 - cfg->damping) / (double)seeds.size());
        for (uint32_t v : seeds) {
            GCHI_CHECK(v < N, GCHI_ERR_INVALID, "ppr_batch_run: seed out of range");
            size_t slot = (size_t)qb * kSeedTable + sn[qb]++;
            sv[slot] = v;
            sq[slot] = lane;
        }
    }
    for (uint32_t qb = 0; qb < nqb; qb++) {  // sort each table by (vertex, query)
        std::vector<std::pair<uint32_t, uint32_t>> t;
        for (uint32_t k = 0; k < sn[qb]; k++) t.push_back({sv[(size_t)qb * kSeedTable + k], sq[(size_t)qb * kSeedTable + k]});
        std::sort(t.begin(), t.end());
        for (uint32_t k = 0; k < sn[qb]; k++) {
            sv[(size_t)qb * kSeedTable + k] = t[k].first;
            sq[(size_t)qb * kSeedTable + k] = t[k].second;
        }
    }
    GCHI_HIP(hipMemcpyAsync(b->seed_v, sv.data(), sv.size() * 4, hipMemcpyHostToDevice, s));
    GCHI_HIP(hipMemcpyAsync(b->seed_q, sq.data(), sq.size() * 4, hipMemcpyHostToDevice, s));
    GCHI_HIP(hipMemcpyAsync(b->seed_n, sn.data(), sn.size() * 4, hipMemcpyHostToDevice, s));
    GCHI_HIP(hipMemcpyAsync(b->tele, tele.data(), tele.size() * 4, hipMemcpyHostToDevice, s));

    const float d = (float)cfg->damping;
    const double stop = cfg->tol * (1.0 - cfg->damping) / cfg->damping;  // residual bound
    // sweeps run in chunks of `check` (even, so a chunk ends in the buffer it
    // started from), each chunk one HIP-graph launch whose last sweep computes
    // the residuals; converged query blocks leave the active list
    const int check = std::max(2, (cfg->check_every > 0 ? cfg->check_every : 4) & ~1);
    const int max_sweeps = cfg->max_sweeps > 0 ? cfg->max_sweeps : 1000;
    std::vector<double> res((size_t)nqb * kQ, 0.0), last((size_t)nqb * kQ, 0.0);
    std::vector<uint32_t> active(nqb + 1);
    for (uint32_t qb = 0; qb < nqb; qb++) active[qb] = qb;
    active[nqb] = nqb;
    GCHI_HIP(hipMemcpyAsync(b->active, active.data(), 4 * active.size(), hipMemcpyHostToDevice, s));
    uint32_t nact = nqb;
    auto read_res = [&]() -> int {
        GCHI_HIP(hipMemcpyAsync(res.data(), b->res, res.size() * 8, hipMemcpyDeviceToHost, s));
        GCHI_HIP(hipStreamSynchronize(s));
        for (uint32_t i = 0; i < nact; i++)
            for (int l = 0; l < kQ; l++) last[(size_t)active[i] * kQ + l] = res[(size_t)active[i] * kQ + l];
        return GCHI_OK;
    };
    auto max_res = [&]() {
        double m = 0.0;
        for (uint32_t q = 0; q < b->nq; q++) m = std::max(m, last[q]);
        return m;
    };
    result->sweeps_bf16 = result->sweeps_fp32 = result->block_sweeps_fp32 = 0;
    const PpArgs a0 = make_args(b, d);
    const dim3 cgrid(std::max(1u, 4096 / std::min(nqb, 64u)), std::min(nqb, 64u)), sgrid(std::min(nqb, 1024u));
    launch_fill_u32(b->seedk, 0u, (size_t)nqb * a0.kwords, s);
    int sweeps = 0;
    b->cur = 0;
    b->fp32 = cfg->bf16_sweeps <= 0;
    if (!b->fp32) {
        uint16_t *r0 = (uint16_t *)b->r16[0], *r1 = (uint16_t *)b->r16[1];
        hipLaunchKernelGGL(ppr_clear_kernel<uint16_t>, cgrid, dim3(256), 0, s, a0, r0, r1, 1);
        hipLaunchKernelGGL(ppr_seed_kernel<uint16_t>, sgrid, dim3(256), 0, s, a0, r0, r1, b->seedk, 1);
        GCHI_LAUNCH_CHECK();
        GCHI_TRY(ppr_capture_chunk(b, 0, check, d));
        double prev = 1e300;
        while (sweeps + check <= max_sweeps && result->sweeps_bf16 + check <= cfg->bf16_sweeps) {
            GCHI_HIP(hipGraphLaunch(b->chunk_exec[0], s));
            sweeps += check;
            result->sweeps_bf16 += check;
            GCHI_TRY(read_res());
            const double m = max_res();
            // leave BF16 once the residual is small or no longer falls (rounding floor)
            if (m <= cfg->bf16_switch_residual || m > 0.7 * prev) break;
            prev = m;
        }
        hipLaunchKernelGGL(ppr_widen_kernel, dim3(65536), dim3(256), 0, s, (const uint16_t *)b->r16[0], b->r32[0],
                           b->state);
        b->fp32 = true;
    }
    // FP32 teleport values of the rows without in-edges in both buffers; of all
    // rows when there was no BF16 phase
    const int whole = cfg->bf16_sweeps <= 0;
    hipLaunchKernelGGL(ppr_clear_kernel<float>, cgrid, dim3(256), 0, s, a0, b->r32[0], b->r32[1], whole);
    hipLaunchKernelGGL(ppr_seed_kernel<float>, sgrid, dim3(256), 0, s, a0, b->r32[0], b->r32[1], b->seedk, whole);
    GCHI_LAUNCH_CHECK();
    GCHI_TRY(ppr_capture_chunk(b, 1, check, d));
    bool converged = false;
    while (sweeps + check <= max_sweeps) {
        GCHI_HIP(hipGraphLaunch(b->chunk_exec[1], s));
        sweeps += check;
        result->sweeps_fp32 += check;
        GCHI_TRY(read_res());
        // retire the query blocks whose every query meets the bound
        uint32_t keep = 0;
        for (uint32_t i = 0; i < nact; i++) {
            const uint32_t qb = active[i];
            double m = 0.0;
            for (int l = 0; l < kQ; l++) m = std::max(m, last[(size_t)qb * kQ + l]);
            if (m > stop) active[keep++] = qb;
        }
        result->block_sweeps_fp32 += (int)nact * check;
        if (keep == 0) {
            converged = true;
            break;
        }
        if (keep != nact) {
            nact = keep;
            active[nqb] = nact;
            GCHI_HIP(hipMemcpyAsync(b->active, active.data(), 4 * nact, hipMemcpyHostToDevice, s));
            GCHI_HIP(hipMemcpyAsync(b->active + nqb, &active[nqb], 4, hipMemcpyHostToDevice, s));
        }
    }
    GCHI_HIP(hipStreamSynchronize(s));
    result->converged = converged ? 1 : 0;
    result->max_residual = max_res();
    if (h_residuals)
        for (uint32_t q = 0; q < b->nq; q++) h_residuals[q] = last[q];
    return GCHI_OK;
}

extern "C" int gchi_ppr_batch_extract(const gchi_ppr_batch *b, uint32_t query, float *d_out, void *stream) {
    GCHI_CHECK(b && d_out && query < b->nq, GCHI_ERR_INVALID, "ppr_batch_extract: bad argument");
    const void *R = b->fp32 ? (const void *)b->r32[b->cur] : b->r16[b->cur];
    hipLaunchKernelGGL(ppr_extract_kernel, dim3(grid_for(b->N, 256, 65536)), dim3(256), 0, as_stream(stream), b->a, R,
                       b->fp32 ? 1 : 0, query, d_out);
    GCHI_LAUNCH_CHECK();
    return GCHI_OK;
}
