// Triangle counting on the degree-ordered graph.
//
// Reference: example_apps/trianglecounting.cpp.  The input is relabelled by
// order_by_degree (src/preprocessing/util/orderbydegree.hpp:58-100): vertices
// ranked by (in+out degree, id), vertexmap[old] = rank; per-vertex triangle
// counts are stored in the new id space as uint32 (<G>_degord.4B.vout,
// trianglecounting.cpp:72) and the total is their sum / 3 (:476-477).
//
// Device form:
//   gchi_tc_prepare : degrees, (degree,id) radix sort -> vertexmap, edges mapped
//       and oriented from lower to higher rank, sorted and deduplicated into an
//       oriented CSR (N+(v): the higher-ranked neighbours of v, ascending).
//   gchi_tc_count   : every triangle a<b<w is found once, at vertex a, as
//       w in N+(a) n N+(b) for b in N+(a).  One wavefront per vertex a.
//       w among the 4096 highest ranks (the core; nearly all wedges of a skewed
//       graph end there): tc_count_core_kernel, rows as bitmaps.
//       The other w by the length of N+(a) without its core entries.  Up to 512
//       (tc_count_tail_kernel): the (b, w in N+(b)) pairs of 64 consecutive b are
//       flattened over the 64 lanes, and each w passes a 4096-bit filter of N+(a)
//       in LDS before it is searched there.  Up to 1024 (tc_count_hash_kernel):
//       every w is looked up in an LDS hash table of N+(a).  Longer
//       (tc_count_kernel): the tail's pairs, each lane binary-searching its w in
//       N+(a).  gchi_tc_count_noalloc has no core (no scratch for its bitmaps): the
//       tail kernel takes rows of up to 64 entries there, the hash kernel the rest.
//       Counts: a, b and w each get +1 per triangle, gathered per wavefront or
//       workgroup and converted to uint32 with an overflow flag.
#include <mutex>

#include "common.hpp"
#include "internal.hpp"

namespace gchi {

constexpr int kTcWaves = 4;
constexpr int kTcLds = 1024;

// Degree keys: (dst << sb) | src with sb = the id field width rounded up to a
// whole radix digit; the id field is wide enough to hold n itself, which marks
// self-loops (and out-of-range ids, reported through err) so that run counting
// skips them.
__global__ void tc_degree_pack(const uint32_t *src, const uint32_t *dst, uint64_t e, uint32_t n, int sb,
                               uint64_t *keys, uint32_t *err) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < e; i += stride) {
        uint32_t s = src[i], d = dst[i];
        if (s >= n || d >= n) atomicOr(err, 1u);
        if (s >= n || d >= n || s == d) s = d = n;
        keys[i] = ((uint64_t)d << sb) | s;
    }
}

__global__ void tc_degree_keys(const uint32_t *deg, uint32_t n, int idb, uint64_t *keys) {
    uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride)
        keys[v] = ((uint64_t)deg[v] << idb) | v;
}

// Ids >= n appear only in the output of a sort whose look-back gave up (the
// caller reports that and discards the result): skipped so that no write leaves
// the arrays.  The same guard is in the two run kernels below.
__global__ void tc_vertexmap(const uint64_t *keys, uint32_t n, int idb, uint32_t *vmap) {
    uint32_t stride = gridDim.x * blockDim.x;
    const uint64_t m = (1ull << idb) - 1ull;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const uint64_t v = keys[i] & m;
        if (v < n) vmap[v] = i;
    }
}

__global__ void tc_orient_keys(const uint32_t *src, const uint32_t *dst, uint64_t e, uint32_t n, const uint32_t *vmap, int idb,
                               uint64_t sentinel, uint64_t *keys) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < e; i += stride) {
        uint32_t s = src[i], d = dst[i];
        if (s == d || s >= n || d >= n) {  // out-of-range ids are reported by tc_degree_pack
            keys[i] = sentinel;
            continue;
        }
        uint32_t a = vmap[s], b = vmap[d];
        uint32_t lo = min(a, b), hi = max(a, b);
        keys[i] = ((uint64_t)lo << idb) | hi;
    }
}

__global__ void tc_unique_flags(const uint64_t *keys, uint64_t e, uint64_t sentinel, uint32_t *flags) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < e; i += stride) {
        uint64_t k = keys[i];
        flags[i] = (k != sentinel && (i == 0 || keys[i - 1] != k)) ? 1u : 0u;
    }
}

// Runs of equal lo = key >> idb in the sorted oriented keys (sentinel keys,
// which sort last, excluded).  lo_start[lo] = pos at the run's first key.
__global__ void tc_lo_run_starts(const uint64_t *keys, const uint32_t *pos, uint64_t e, int idb, uint64_t sentinel,
                                 uint32_t n, uint32_t *lo_start) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < e; i += stride) {
        const uint64_t k = keys[i];
        if (k == sentinel) continue;
        const uint64_t lo = k >> idb;
        if (lo >= n) continue;
        if (i == 0 || (keys[i - 1] >> idb) != lo) lo_start[lo] = pos[i];
    }
}

// adj[pos] = hi of every unique key; at a run's last key, lo_count[lo] = the
// unique keys of the run (no atomics: one writer per run).
__global__ void tc_scatter_unique(const uint64_t *keys, const uint32_t *flags, const uint32_t *pos, uint64_t e,
                                  int idb, uint64_t sentinel, uint32_t n, const uint32_t *lo_start, uint32_t *adj,
                                  uint32_t *lo_count) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint64_t m = (1ull << idb) - 1ull;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < e; i += stride) {
        const uint64_t k = keys[i];
        if (k == sentinel) continue;
        const uint64_t lo = k >> idb;
        if (lo >= n) continue;
        const uint32_t f = flags[i], p = pos[i];
        if (f) adj[p] = (uint32_t)(k & m);
        const bool last = i + 1 == e || keys[i + 1] == sentinel || (keys[i + 1] >> idb) != lo;
        if (last) lo_count[lo] = p + f - lo_start[lo];
    }
}

// Position of x in the ascending a[lo, hi), or -1.
GCHI_DEV int bsearch_u32(const uint32_t *a, uint32_t lo, uint32_t hi, uint32_t x) {
    while (lo < hi) {
        uint32_t mid = (lo + hi) >> 1;
        uint32_t v = a[mid];
        if (v == x) return (int)mid;
        if (v < x)
            lo = mid + 1;
        else
            hi = mid;
    }
    return -1;
}

// end[v] = where the row ends for this kernel and the tail kernel: off[v + 1], or
// the row's first core entry.
__global__ __launch_bounds__(kTcWaves *kWave) void tc_count_kernel(const uint32_t *__restrict__ off,
                                                                   const uint32_t *__restrict__ end,
                                                                   const uint32_t *__restrict__ adj, uint32_t n,
                                                                   uint32_t min_da, unsigned long long *cnt,
                                                                   unsigned long long *total) {
    __shared__ uint32_t sA[kTcWaves][kTcLds];
    __shared__ uint32_t sW[kTcWaves][kTcLds];  // triangles found per position of N+(a) (the w credit)
    __shared__ uint32_t sPre[kTcWaves][kWave];
    __shared__ uint32_t sBeg[kTcWaves][kWave];
    __shared__ uint32_t sCnt[kTcWaves][kWave];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    // A static scan, 64 vertices per step, picks the vertices above min_da (no
    // work counter: the few long rows would not pay for a ticket per vertex).
    const uint64_t step = (uint64_t)gridDim.x * kTcWaves * kWave;
    for (uint64_t base = ((uint64_t)blockIdx.x * kTcWaves + wave) * kWave; base < n; base += step) {
        const uint64_t v = base + lane;
        const uint32_t dv = v < n ? end[v] - off[v] : 0u;
        uint64_t todo = __ballot(dv >= 2 && dv > min_da);
        while (todo) {
        const uint32_t a = (uint32_t)base + (uint32_t)__builtin_ctzll(todo);
        todo &= todo - 1;
        const uint32_t ab = off[a], da = end[a] - ab;
        const uint32_t *A = adj + ab;
        const bool lds = da <= (uint32_t)kTcLds;
        if (lds)
            for (uint32_t k = lane; k < da; k += kWave) {
                sA[wave][k] = A[k];
                sW[wave][k] = 0u;
            }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const uint32_t *As = lds ? sA[wave] : A;
        unsigned long long acc_a = 0;
        for (uint32_t bc = 0; bc + 1 < da; bc += kWave) {
            const uint32_t k = bc + lane;
            const bool valid = k < da;
            uint32_t b = valid ? As[k] : 0u;
            uint32_t bb = valid ? off[b] : 0u;
            uint32_t lb = valid ? end[b] - bb : 0u;
            uint32_t pre = lb;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                uint32_t t = __shfl_up(pre, o, kWave);
                if (lane >= o) pre += t;
            }
            const uint32_t tot = __shfl(pre, kWave - 1, kWave);
            sPre[wave][lane] = pre;
            sBeg[wave][lane] = bb;
            sCnt[wave][lane] = 0;
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            for (uint32_t p = lane; p < tot; p += kWave) {
                uint32_t lo = 0, hi = kWave - 1;
                while (lo < hi) {
                    uint32_t mid = (lo + hi) >> 1;
                    if (sPre[wave][mid] > p)
                        hi = mid;
                    else
                        lo = mid + 1;
                }
                const uint32_t j = lo;
                const uint32_t excl = j ? sPre[wave][j - 1] : 0u;
                const uint32_t w = adj[sBeg[wave][j] + (p - excl)];
                // w > b_j > a; N+(a) is ascending, b_j sits at index bc + j
                const int kw = bsearch_u32(As, bc + j + 1, da, w);
                if (kw >= 0) {
                    if (lds)
                        atomicAdd(&sW[wave][kw], 1u);
                    else
                        atomicAdd(&cnt[w], 1ull);
                    atomicAdd(&sCnt[wave][j], 1u);
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            const uint32_t c = valid ? sCnt[wave][lane] : 0u;
            if (c) atomicAdd(&cnt[b], (unsigned long long)c);
            acc_a += c;
            __builtin_amdgcn_wave_barrier();
        }
        if (lds) {  // one global atomic per w of N+(a) that closed a triangle
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            for (uint32_t k = lane; k < da; k += kWave) {
                const uint32_t cw = sW[wave][k];
                if (cw) atomicAdd(&cnt[sA[wave][k]], (unsigned long long)cw);
            }
        }
        acc_a = wave_sum(acc_a);
        if (lane == 0 && acc_a) {
            atomicAdd(&cnt[a], acc_a);
            atomicAdd(total, acc_a);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        }
    }
}

// Inclusive scans over the wavefront (sum; maximum), in six steps.
template <int CTRL, int ROWS>
GCHI_DEV uint32_t tc_dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
}
GCHI_DEV uint32_t tc_scan_sum(uint32_t v) {
    v += tc_dpp<0x111, 0xf>(v);  // row_shr:1
    v += tc_dpp<0x112, 0xf>(v);  // row_shr:2
    v += tc_dpp<0x114, 0xf>(v);  // row_shr:4
    v += tc_dpp<0x118, 0xf>(v);  // row_shr:8
    v += tc_dpp<0x142, 0xa>(v);  // row_bcast:15
    v += tc_dpp<0x143, 0xc>(v);  // row_bcast:31
    return v;
}
GCHI_DEV uint32_t tc_scan_max(uint32_t v) {
    v = max(v, tc_dpp<0x111, 0xf>(v));
    v = max(v, tc_dpp<0x112, 0xf>(v));
    v = max(v, tc_dpp<0x114, 0xf>(v));
    v = max(v, tc_dpp<0x118, 0xf>(v));
    v = max(v, tc_dpp<0x142, 0xa>(v));
    v = max(v, tc_dpp<0x143, 0xc>(v));
    return v;
}

GCHI_DEV void tc_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The vertices of wavefront w are n-1-w, n-1-w-nw, ... (nw wavefronts): the work
// per vertex changes slowly with its rank, so every wavefront gets a like share
// without tickets (which took 146 of 1105 us per wavefront in the core kernel).
// Lane l holds the row bounds of the l-th of the next 64 vertices.

// |N+(a)| in [2, max_da]: N+(a) in LDS with a bit filter of its ids, the pairs of
// 64 b at a time in flattened order, kTcTailStep pairs per lane in
// flight.  A pair's b comes from marks in LDS at the first pair of every b and a
// maximum scan.  Bound: vector instructions (about 30 per 64 pairs) and, in
// sparse graphs, the three dependent loads per vertex (row, b's bounds, w).
// Short rows keep all lanes busy this way: the form before it, one b at a time
// against a hash table, took 882 us for the tails of R-MAT scale 19 (75M pairs),
// this one 172 us.
constexpr int kTcTailWaves = 4;
constexpr uint32_t kTcTailMax = 512;
constexpr uint32_t kTcTailMaxWhole = 64;  // without a core (see tc_count_hash_kernel)
constexpr int kTcTailStep = 4;

GCHI_DEV uint32_t tc_filter(uint32_t x) { return (x ^ (x >> 12)) & 4095u; }

__global__ __launch_bounds__(kTcTailWaves *kWave) void tc_count_tail_kernel(const uint32_t *__restrict__ off,
                                                                            const uint32_t *__restrict__ end,
                                                                            const uint32_t *__restrict__ adj,
                                                                            uint32_t n, uint32_t max_da,
                                                                            unsigned long long *cnt,
                                                                            unsigned long long *total) {
    __shared__ uint32_t s_a[kTcTailWaves][kTcTailMax];    // N+(a), ascending
    __shared__ uint32_t s_c[kTcTailWaves][kTcTailMax];    // credits of its entries
    __shared__ uint32_t s_bits[kTcTailWaves][4096 / 32];
    __shared__ uint32_t s_mark[kTcTailWaves][kTcTailStep * kWave];
    __shared__ uint32_t s_hit[kTcTailWaves][kWave];
    __shared__ unsigned long long s_total;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    uint32_t *A = s_a[wave], *C = s_c[wave], *bits = s_bits[wave], *mark = s_mark[wave], *hitc = s_hit[wave];
    if (threadIdx.x == 0) s_total = 0;
    __syncthreads();
    unsigned long long acc_total = 0;
    const uint64_t nw = (uint64_t)gridDim.x * kTcTailWaves;
    for (uint64_t i0 = (uint64_t)blockIdx.x * kTcTailWaves + wave; i0 < n; i0 += nw * kWave) {
        const uint64_t mine = i0 + nw * lane;
        const uint32_t va = mine < n ? n - 1 - (uint32_t)mine : 0u;
        const uint32_t vb = mine < n ? off[va] : 0u, ve = mine < n ? end[va] : 0u;
        uint64_t todo = __ballot(ve - vb >= 2 && ve - vb <= max_da);
        while (todo) {
            const int l = __builtin_ctzll(todo);
            todo &= todo - 1;
            const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)va, l);
            const uint32_t ab = (uint32_t)__builtin_amdgcn_readlane((int)vb, l);
            const uint32_t da = (uint32_t)__builtin_amdgcn_readlane((int)ve, l) - ab;
            bits[lane] = bits[lane + kWave] = 0u;
            tc_lds_sync();
            for (uint32_t k = lane; k < da; k += kWave) {
                const uint32_t x = adj[ab + k], h = tc_filter(x);
                A[k] = x;
                C[k] = 0u;
                atomicOr(&bits[h >> 5], 1u << (h & 31));
            }
            tc_lds_sync();
            uint32_t acc_a = 0;
            for (uint32_t bc = 0; bc + 1 < da; bc += kWave) {  // the last neighbour has no w above it
                const bool valid = bc + lane + 1 < da;
                const uint32_t b = valid ? A[bc + lane] : 0u;
                const uint32_t bb = valid ? off[b] : 0u;
                const uint32_t lb = valid ? end[b] - bb : 0u;
                const uint32_t pre = tc_scan_sum(lb);
                const uint32_t tot = (uint32_t)__builtin_amdgcn_readlane((int)pre, kWave - 1);
                const uint32_t first = pre - lb;  // b's first pair
                const uint32_t shift = bb - first;
                hitc[lane] = 0u;
                uint32_t carry = 0;  // 1 + lane of the b that the last pair so far belongs to
                for (uint32_t p0 = 0; p0 < tot; p0 += kTcTailStep * kWave) {
#pragma unroll
                    for (int u = 0; u < kTcTailStep; u++) mark[u * kWave + lane] = 0u;
                    tc_lds_sync();
                    if (lb && first - p0 < (uint32_t)(kTcTailStep * kWave)) mark[first - p0] = (uint32_t)lane + 1;
                    tc_lds_sync();
                    uint32_t w[kTcTailStep], j[kTcTailStep];
#pragma unroll
                    for (int u = 0; u < kTcTailStep; u++) {
                        const uint32_t m = max(tc_scan_max(mark[u * kWave + lane]), carry);
                        carry = (uint32_t)__builtin_amdgcn_readlane((int)m, kWave - 1);
                        j[u] = m - 1;
                        const uint32_t p = p0 + u * kWave + lane;
                        const uint32_t at = (uint32_t)__shfl((int)shift, (int)j[u], kWave) + p;
                        w[u] = p < tot ? adj[at] : n;
                    }
#pragma unroll
                    for (int u = 0; u < kTcTailStep; u++) {
                        const uint32_t h = tc_filter(w[u]);
                        if (w[u] < n && ((bits[h >> 5] >> (h & 31)) & 1u)) {
                            // w > b, which is entry bc + j of N+(a)
                            const int k = bsearch_u32(A, bc + j[u] + 1, da, w[u]);
                            if (k >= 0) {
                                atomicAdd(&C[k], 1u);
                                atomicAdd(&hitc[j[u]], 1u);
                            }
                        }
                    }
                    tc_lds_sync();
                }
                tc_lds_sync();
                const uint32_t c = hitc[lane];
                if (c) atomicAdd(&C[bc + lane], c);
                acc_a += c;
                tc_lds_sync();
            }
            for (uint32_t k = lane; k < da; k += kWave) {
                const uint32_t c = C[k];
                if (c) atomicAdd(&cnt[A[k]], (unsigned long long)c);
            }
            acc_a = wave_sum(acc_a);  // at most kTcTailMax^2 / 2
            if (lane == 0 && acc_a) atomicAdd(&cnt[a], (unsigned long long)acc_a);
            acc_total += acc_a;
            tc_lds_sync();
        }
    }
    if (lane == 0 && acc_total) atomicAdd(&s_total, acc_total);
    __syncthreads();
    if (threadIdx.x == 0 && s_total) atomicAdd(total, s_total);
}

// |N+(a)| in (min_da, kTcHashMax]: one wavefront puts N+(a) into an LDS hash table
// (open addressing, linear probing, at most half full), then walks b in N+(a) one
// at a time and looks up every w in N+(b) lane-wide, kTcInflight w per lane in
// flight.  w's and b's credits go to their slots (16-bit halves of LDS words: at
// most 2|N+(a)| per slot) and are added to the global counts once per a.
// Bound: LDS probes, one or two per pair whether it closes a triangle or not; the
// tail kernel pays about 30 instructions per 64 pairs and a binary search per
// triangle.  So the line between them (min_da) lies where pairs close.  With the
// core split off few do, and the tail kernel keeps what it holds (kTcTailMax; R-MAT
// scale 21 with 14.9M edges: 2.5 ms, 3.0 with the line at 64).  Without a core:
//   us at line           64      128     256     512
//   clique of 150       190      280     201     198
//   clique of 300       389      472     867     757
//   clique of 600       924    1,011   1,404   3,114
//   R-MAT scale 17    1,360    1,318   1,289   1,174
//   R-MAT scale 19    5,741    5,255   5,378   5,707
//   rows of 90, few  17,300    7,189   6,934   6,896
// and 64 is the only one that is nowhere far slower than the hash table alone
// (204, 395, 927, 1,409, 6,169 and 16,452 us).  Searched for every pair from 513
// entries on, the clique of 600 took 225 ms and R-MAT scale 19 36.8.
// More workgroups than fit, so that the hardware evens out rows of different
// lengths (6 / 12 / 24 / 48 per CU: 12.3 / 12.5 / 11.2 / 12.0 ms for 40,000 rows of
// about 300).
constexpr int kTcHashWaves = 4;
constexpr uint32_t kTcHashSlots = 2048;
constexpr uint32_t kTcHashMax = kTcHashSlots / 2;
constexpr uint32_t kTcEmpty = 0xffffffffu;
constexpr unsigned kTcHashGrid = 24;  // workgroups per CU
constexpr int kTcInflight = 8;  // w loads per lane in flight (one memory round trip per 512 w)

GCHI_DEV uint32_t tc_slot(uint32_t w, int sh) { return (w * 2654435761u) >> sh; }

GCHI_DEV int tc_find(const uint32_t *keys, uint32_t mask, int sh, uint32_t w) {
    uint32_t h = tc_slot(w, sh);
    for (;;) {
        const uint32_t k = keys[h];
        if (k == w) return (int)h;
        if (k == kTcEmpty) return -1;
        h = (h + 1) & mask;
    }
}

GCHI_DEV void tc_credit(uint32_t *cw, uint32_t slot, uint32_t c) { atomicAdd(&cw[slot >> 1], c << ((slot & 1) * 16)); }

// Entry `lane` of N+(b_j) (b_j, its start and length in lane j of b/bb/lb), or
// kTcEmpty past the list; the load is issued at an in-bounds address either way.
GCHI_DEV uint32_t tc_first_w(const uint32_t *adj, uint32_t bb, uint32_t lb, uint32_t j, int lane) {
    const uint32_t bbj = (uint32_t)__builtin_amdgcn_readlane((int)bb, (int)j);
    const uint32_t lbj = (uint32_t)__builtin_amdgcn_readlane((int)lb, (int)j);
    const uint32_t v = adj[lbj ? bbj + min((uint32_t)lane, lbj - 1) : 0u];
    return (uint32_t)lane < lbj ? v : kTcEmpty;
}

// Triangles (a, b_j, w) for w in N+(b_j): w0 holds the list's first 64
// entries, the rest are loaded here; each w found in the table is credited,
// and b_j once with the wavefront's total.  Returns that total.
GCHI_DEV uint32_t tc_count_b(const uint32_t *adj, const uint32_t *keys, uint32_t *cw, uint32_t mask, int sh,
                             uint32_t b, uint32_t bb, uint32_t lb, uint32_t j, uint32_t w0, int lane) {
    const uint32_t bj = (uint32_t)__builtin_amdgcn_readlane((int)b, (int)j);
    const uint32_t bbj = (uint32_t)__builtin_amdgcn_readlane((int)bb, (int)j);
    const uint32_t lbj = (uint32_t)__builtin_amdgcn_readlane((int)lb, (int)j);
    const uint32_t *B = adj + bbj;
    uint32_t hits = 0;
    if (w0 != kTcEmpty) {
        const int h = tc_find(keys, mask, sh, w0);
        if (h >= 0) {
            tc_credit(cw, (uint32_t)h, 1u);
            hits++;
        }
    }
    for (uint32_t t = kWave + lane; t < lbj; t += kTcInflight * kWave) {
        uint32_t w[kTcInflight];
#pragma unroll
        for (int q = 0; q < kTcInflight; q++) {
            const uint32_t tq = t + q * kWave;
            w[q] = tq < lbj ? B[tq] : kTcEmpty;
        }
#pragma unroll
        for (int q = 0; q < kTcInflight; q++) {
            if (w[q] == kTcEmpty) continue;
            const int h = tc_find(keys, mask, sh, w[q]);
            if (h >= 0) {
                tc_credit(cw, (uint32_t)h, 1u);
                hits++;
            }
        }
    }
    hits = wave_sum(hits);
    if (hits && lane == 0) tc_credit(cw, (uint32_t)tc_find(keys, mask, sh, bj), hits);
    return hits;
}

__global__ __launch_bounds__(kTcHashWaves *kWave) void tc_count_hash_kernel(const uint32_t *__restrict__ off,
                                                                            const uint32_t *__restrict__ end,
                                                                            const uint32_t *__restrict__ adj,
                                                                            uint32_t n, uint32_t min_da,
                                                                            unsigned long long *cnt,
                                                                            unsigned long long *total) {
    __shared__ uint32_t sKey[kTcHashWaves][kTcHashSlots];
    __shared__ uint32_t sCw[kTcHashWaves][kTcHashSlots / 2];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    uint32_t *keys = sKey[wave];
    uint32_t *cw = sCw[wave];
    unsigned long long acc_total = 0;
    const uint64_t nw = (uint64_t)gridDim.x * kTcHashWaves;
    for (uint64_t i0 = (uint64_t)blockIdx.x * kTcHashWaves + wave; i0 < n; i0 += nw * kWave) {
        const uint64_t mine = i0 + nw * lane;
        const uint32_t va = mine < n ? n - 1 - (uint32_t)mine : 0u;
        const uint32_t vb = mine < n ? off[va] : 0u, ve = mine < n ? end[va] : 0u;
        uint64_t todo = __ballot(ve - vb > min_da && ve - vb <= kTcHashMax);
        while (todo) {
            const int l = __builtin_ctzll(todo);
            todo &= todo - 1;
            const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)va, l);
            const uint32_t ab = (uint32_t)__builtin_amdgcn_readlane((int)vb, l);
            const uint32_t da = (uint32_t)__builtin_amdgcn_readlane((int)ve, l) - ab;
            const uint32_t want = 4 * da;  // slots: pow2 >= 4 da, at most kTcHashSlots
            const int lg = min(32 - __clz((int)(want - 1)), 11);
            const uint32_t S = 1u << lg, mask = S - 1;
            const int sh = 32 - lg;
            for (uint32_t k = lane; k < S; k += kWave) keys[k] = kTcEmpty;
            for (uint32_t k = lane; k < S / 2; k += kWave) cw[k] = 0u;
            tc_lds_sync();
            const uint32_t *A = adj + ab;
            for (uint32_t k = lane; k < da; k += kWave) {
                const uint32_t x = A[k];
                uint32_t h = tc_slot(x, sh);
                while (atomicCAS(&keys[h], kTcEmpty, x) != kTcEmpty) h = (h + 1) & mask;
            }
            tc_lds_sync();
            uint32_t acc_a = 0;
            // the last element of N+(a) closes no triangle here (no w above it)
            for (uint32_t bc = 0; bc + 1 < da; bc += kWave) {
                const uint32_t k = bc + lane;
                const bool valid = k + 1 < da;
                const uint32_t b = valid ? A[k] : 0u;
                const uint32_t bb = valid ? off[b] : 0u;
                const uint32_t lb = valid ? end[b] - bb : 0u;
                const uint32_t nb = min((uint32_t)kWave, da - 1 - bc);
                // The first 64 entries of N+(b_j) are loaded one b ahead (slots w2[0],
                // w2[1] in turn), so that b_j's probes overlap b_{j+1}'s loads.
                uint32_t w2[2];
                w2[0] = tc_first_w(adj, bb, lb, 0, lane);
                for (uint32_t j0 = 0; j0 < nb; j0 += 2) {  // loads unconditional (clamped j), uses not
                    w2[1] = tc_first_w(adj, bb, lb, min(j0 + 1, nb - 1), lane);
                    acc_a += tc_count_b(adj, keys, cw, mask, sh, b, bb, lb, j0, w2[0], lane);
                    w2[0] = tc_first_w(adj, bb, lb, min(j0 + 2, nb - 1), lane);
                    if (j0 + 1 < nb) acc_a += tc_count_b(adj, keys, cw, mask, sh, b, bb, lb, j0 + 1, w2[1], lane);
                }
            }
            tc_lds_sync();
            for (uint32_t k = lane; k < S; k += kWave) {
                const uint32_t key = keys[k];
                const uint32_t c = (cw[k >> 1] >> ((k & 1) * 16)) & 0xffffu;
                if (key != kTcEmpty && c) atomicAdd(&cnt[key], (unsigned long long)c);
            }
            if (lane == 0 && acc_a) atomicAdd(&cnt[a], (unsigned long long)acc_a);
            acc_total += acc_a;
            tc_lds_sync();
        }
    }
    if (lane == 0 && acc_total) atomicAdd(total, acc_total);
}

// ---- the core: triangles whose highest vertex w is among the kTcCore highest ranks ----
// In a skewed graph nearly all wedges end there (96% at R-MAT scale 19), and the
// rows that make them are dense in it, so a row's core entries are a bitmap of
// kTcCore bits, 64 per lane: the w of (a, b) are one AND, their number one
// popcount, and the credits of w vertical counters in registers (bit planes
// summed with carry-save adders, flushed every 2^kTcPlanes bitmaps).  Bitmaps
// are kept for the rows with more than kTcList core entries (one per lane: 752 us
// at R-MAT scale 19, 811 with 128) of the highest ranks; the entries of other
// rows are tested one by one against N+(a)'s bitmap in LDS.
// Bound: vector instructions (about 25 per bitmap) and the L2 reads of the
// bitmaps (512 bytes each; two sets of eight rows take turns so that one is in
// flight).  R-MAT scale 19, 7.7M edges, 1.71G wedges: 752 us, and 34 for the
// workgroups' credits; the hash table that looked up every wedge took 6312 us.
constexpr uint32_t kTcCore = 4096;
constexpr uint32_t kTcCoreWords = kTcCore / 32;
constexpr uint32_t kTcList = 64;
constexpr uint32_t kTcMapRows = 1u << 18;   // at most 128 MiB of bitmaps
constexpr uint32_t kTcNear = 16384;         // ranks whose b and w credits are counted in LDS
constexpr int kTcCoreThreads = 512;
constexpr int kTcCoreWaves = kTcCoreThreads / kWave;
constexpr int kTcPlanes = 12;

// end[v] = first entry of v's row in the core (rank >= base).
__global__ void tc_core_split(const uint32_t *__restrict__ off, const uint32_t *__restrict__ adj, uint32_t n,
                              uint32_t base, uint32_t *__restrict__ end) {
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride) {
        uint32_t lo = off[v], hi = off[v + 1];
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (adj[mid] >= base) hi = mid;
            else lo = mid + 1;
        }
        end[v] = lo;
    }
}

// One wavefront per row v = first + r with more than kTcList core entries: its bitmap.
__global__ __launch_bounds__(256) void tc_core_maps(const uint32_t *__restrict__ off, const uint32_t *__restrict__ adj,
                                                    const uint32_t *__restrict__ end, uint32_t first, uint32_t rows,
                                                    uint32_t base, uint2 *__restrict__ maps) {
    __shared__ uint32_t s_bits[256 / kWave][kTcCoreWords];
    const int lane = threadIdx.x & (kWave - 1);
    uint32_t *bits = s_bits[threadIdx.x / kWave];
    const uint32_t nw = gridDim.x * (256 / kWave);
    for (uint32_t r = blockIdx.x * (256 / kWave) + threadIdx.x / kWave; r < rows; r += nw) {
        const uint32_t b = end[first + r], e = off[first + r + 1];
        if (e - b <= kTcList) continue;
        bits[lane] = bits[lane + kWave] = 0u;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (uint32_t k = b + lane; k < e; k += kWave) {
            const uint32_t c = adj[k] - base;
            atomicOr(&bits[c >> 5], 1u << (c & 31));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        maps[(uint64_t)r * kWave + lane] = make_uint2(bits[2 * lane], bits[2 * lane + 1]);
        __builtin_amdgcn_wave_barrier();
    }
}

// sum and carry of three words
GCHI_DEV void tc_csa(uint32_t &s, uint32_t &c, uint32_t x, uint32_t y, uint32_t z) {
    const uint32_t u = x ^ y;
    c = (x & y) | (u & z);
    s = u ^ z;
}

// Adds eight words to the bit planes.
GCHI_DEV void tc_planes_add(uint32_t (&p)[kTcPlanes], const uint32_t (&x)[8]) {
    uint32_t a, b, c, d, e;
    tc_csa(p[0], a, p[0], x[0], x[1]);
    tc_csa(p[0], b, p[0], x[2], x[3]);
    tc_csa(p[1], c, p[1], a, b);
    tc_csa(p[0], a, p[0], x[4], x[5]);
    tc_csa(p[0], b, p[0], x[6], x[7]);
    tc_csa(p[1], d, p[1], a, b);
    tc_csa(p[2], e, p[2], c, d);
#pragma unroll
    for (int k = 3; k < kTcPlanes; k++) {
        const uint32_t t = p[k] & e;
        p[k] ^= e;
        e = t;
    }
}

// Eight bitmap rows in flight: rows of lanes j (of their b), `some` of them.
struct TcRows {
    uint32_t x0[8], x1[8], j[8], some;
};

GCHI_DEV void tc_rows_load(TcRows &g, uint64_t &m, uint32_t b, uint32_t first, const uint2 *__restrict__ maps,
                           int lane) {
    g.some = (uint32_t)__popcll(m);
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const bool on = (uint32_t)u < g.some;  // wavefront-uniform
        g.j[u] = on ? (uint32_t)__builtin_ctzll(m) : 0u;
        m &= m - (on ? 1ull : 0ull);
        g.x0[u] = g.x1[u] = 0u;
        if (on) {
            const uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)b, (int)g.j[u]) - first;
            const uint2 w = maps[(uint64_t)r * kWave + lane];
            g.x0[u] = w.x;
            g.x1[u] = w.y;
        }
    }
}

// ANDs the rows with N+(a) (a0, a1), adds them to the planes, and gives lane
// j[u] the number of common bits of its row in tb.
GCHI_DEV void tc_rows_count(TcRows &g, uint32_t a0, uint32_t a1, uint32_t (&p0)[kTcPlanes], uint32_t (&p1)[kTcPlanes],
                            uint32_t &tb, int lane) {
    uint32_t sum[4];
#pragma unroll
    for (int u = 0; u < 8; u++) {
        g.x0[u] &= a0;
        g.x1[u] &= a1;
    }
    tc_planes_add(p0, g.x0);
    tc_planes_add(p1, g.x1);
#pragma unroll
    for (int u = 0; u < 4; u++)  // two counts (at most kTcCore each) per sum
        sum[u] = tc_scan_sum((uint32_t)(__popc(g.x0[2 * u]) + __popc(g.x1[2 * u])) +
                             ((uint32_t)(__popc(g.x0[2 * u + 1]) + __popc(g.x1[2 * u + 1])) << 16));
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const uint32_t both = (uint32_t)__builtin_amdgcn_readlane((int)sum[u / 2], kWave - 1);
        const uint32_t c = u & 1 ? both >> 16 : both & 0xffffu;
        if ((uint32_t)u < g.some) tb = (uint32_t)lane == g.j[u] ? c : tb;
    }
}

// Eight short rows in flight, up to kTcList entries each.
struct TcLists {
    uint32_t w[8], j[8], some;
};
static_assert(kTcList <= kWave, "one entry per lane");

GCHI_DEV void tc_lists_load(TcLists &g, uint64_t &m, uint32_t bs, uint32_t lb, const uint32_t *__restrict__ adj,
                            uint32_t n, int lane) {
    g.some = (uint32_t)__popcll(m);
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const bool on = (uint32_t)u < g.some;
        g.j[u] = on ? (uint32_t)__builtin_ctzll(m) : 0u;
        m &= m - (on ? 1ull : 0ull);
        const uint32_t beg = (uint32_t)__builtin_amdgcn_readlane((int)bs, (int)g.j[u]);
        const uint32_t len = on ? (uint32_t)__builtin_amdgcn_readlane((int)lb, (int)g.j[u]) : 0u;
        g.w[u] = (uint32_t)lane < len ? adj[beg + lane] : n;
    }
}

GCHI_DEV void tc_lists_count(const TcLists &g, const uint32_t *bits, uint32_t *core, uint32_t base, uint32_t n,
                             uint32_t &tb, int lane) {
#pragma unroll
    for (int u = 0; u < 8; u++) {
        bool hit = false;
        if (g.w[u] < n) {
            const uint32_t c = g.w[u] - base;
            hit = (bits[c >> 5] >> (c & 31)) & 1u;
            if (hit) atomicAdd(&core[c], 1u);
        }
        const uint32_t hits = (uint32_t)__popcll(__ballot(hit));
        if ((uint32_t)u < g.some) tb = (uint32_t)lane == g.j[u] ? hits : tb;
    }
}

__global__ __launch_bounds__(kTcCoreThreads, 4) void tc_count_core_kernel(
    const uint32_t *__restrict__ off, const uint32_t *__restrict__ adj, const uint32_t *__restrict__ end, uint32_t n,
    uint32_t base, uint32_t near, uint32_t first, const uint2 *__restrict__ maps, unsigned long long *cnt,
    unsigned long long *total, uint32_t *__restrict__ slab) {
    __shared__ uint32_t s_near[kTcNear];  // credits of the ranks from near
    __shared__ uint32_t s_bits[kTcCoreWaves][kTcCoreWords];
    __shared__ unsigned long long s_total;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    uint32_t *bits = s_bits[wave];
    uint32_t *core = s_near + (base - near);
    for (uint32_t k = threadIdx.x; k < kTcNear; k += kTcCoreThreads) s_near[k] = 0u;
    if (threadIdx.x == 0) s_total = 0;
    __syncthreads();
    uint32_t p0[kTcPlanes], p1[kTcPlanes];
#pragma unroll
    for (int k = 0; k < kTcPlanes; k++) p0[k] = p1[k] = 0u;
    uint32_t held = 0;  // bitmaps in the planes
    auto flush = [&]() {
        for (uint32_t i = 0; i < 32; i++) {
            uint32_t c0 = 0, c1 = 0;
#pragma unroll
            for (int k = 0; k < kTcPlanes; k++) {
                c0 |= ((p0[k] >> i) & 1u) << k;
                c1 |= ((p1[k] >> i) & 1u) << k;
            }
            if (c0) atomicAdd(&core[lane * 64 + i], c0);
            if (c1) atomicAdd(&core[lane * 64 + 32 + i], c1);
        }
#pragma unroll
        for (int k = 0; k < kTcPlanes; k++) p0[k] = p1[k] = 0u;
        held = 0;
    };
    unsigned long long acc_total = 0;
    const uint64_t nw = (uint64_t)gridDim.x * kTcCoreWaves;
    for (uint64_t i0 = (uint64_t)blockIdx.x * kTcCoreWaves + wave; i0 < n; i0 += nw * kWave) {
        const uint64_t mine = i0 + nw * lane;
        const uint32_t va = mine < n ? n - 1 - (uint32_t)mine : 0u;
        const uint32_t vb = mine < n ? off[va] : 0u, vc = mine < n ? end[va] : 0u, ve = mine < n ? off[va + 1] : 0u;
        uint64_t todo = __ballot(ve - vb >= 2 && vc != ve);
        while (todo) {
            const int l = __builtin_ctzll(todo);
            todo &= todo - 1;
            const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)va, l);
            const uint32_t ab = (uint32_t)__builtin_amdgcn_readlane((int)vb, l);
            const uint32_t ac = (uint32_t)__builtin_amdgcn_readlane((int)vc, l);
            const uint32_t ae = (uint32_t)__builtin_amdgcn_readlane((int)ve, l);
            uint32_t bnext = ab + lane + 1 < ae ? adj[ab + lane] : 0u;
            bits[lane] = bits[lane + kWave] = 0u;
            tc_lds_sync();
            for (uint32_t k = ac + lane; k < ae; k += kWave) {
                const uint32_t c = adj[k] - base;
                atomicOr(&bits[c >> 5], 1u << (c & 31));
            }
            tc_lds_sync();
            const uint32_t a0 = bits[2 * lane], a1 = bits[2 * lane + 1];
            uint32_t acc_a = 0;  // per lane: at most kTcCore per 64 neighbours of a
            for (uint32_t bc = ab; bc + 1 < ae; bc += kWave) {  // the last neighbour has no w above it
                const bool valid = bc + lane + 1 < ae;
                const uint32_t b = bnext;
                const uint32_t bs = valid ? end[b] : 0u;
                const uint32_t lb = valid ? off[b + 1] - bs : 0u;
                bnext = bc + kWave + lane + 1 < ae ? adj[bc + kWave + lane] : 0u;
                const bool mapped = lb > kTcList && b >= first;
                uint32_t tb = 0;  // triangles (a, b of this lane, w)
                uint64_t m = __ballot(mapped);
                if (m) {  // two sets of rows take turns: one loads while the other is counted
                    TcRows ga, gb;
                    tc_rows_load(ga, m, b, first, maps, lane);
                    for (;;) {
                        tc_rows_load(gb, m, b, first, maps, lane);
                        tc_rows_count(ga, a0, a1, p0, p1, tb, lane);
                        held += 8;
                        if (!gb.some) break;
                        tc_rows_load(ga, m, b, first, maps, lane);
                        tc_rows_count(gb, a0, a1, p0, p1, tb, lane);
                        held += 8;
                        if (!ga.some) break;
                    }
                    if (held > (1u << kTcPlanes) - 1 - kWave - 8) flush();  // room for the next 64 neighbours
                }
                m = __ballot(valid && !mapped && lb != 0 && lb <= kTcList);
                if (m) {
                    TcLists ga, gb;
                    tc_lists_load(ga, m, bs, lb, adj, n, lane);
                    for (;;) {
                        tc_lists_load(gb, m, bs, lb, adj, n, lane);
                        tc_lists_count(ga, bits, core, base, n, tb, lane);
                        if (!gb.some) break;
                        tc_lists_load(ga, m, bs, lb, adj, n, lane);
                        tc_lists_count(gb, bits, core, base, n, tb, lane);
                        if (!ga.some) break;
                    }
                }
                m = __ballot(valid && !mapped && lb > kTcList);  // long rows below the bitmapped ranks
                while (m) {
                    const int j = __builtin_ctzll(m);
                    m &= m - 1;
                    const uint32_t beg = (uint32_t)__builtin_amdgcn_readlane((int)bs, j);
                    const uint32_t len = (uint32_t)__builtin_amdgcn_readlane((int)lb, j);
                    uint32_t hits = 0;
                    for (uint32_t k = lane; k - lane < len; k += kWave) {
                        bool hit = false;
                        if (k < len) {
                            const uint32_t c = adj[beg + k] - base;
                            hit = (bits[c >> 5] >> (c & 31)) & 1u;
                            if (hit) atomicAdd(&core[c], 1u);
                        }
                        hits += (uint32_t)__popcll(__ballot(hit));
                    }
                    tb = lane == j ? hits : tb;
                }
                if (tb) {
                    if (b >= near) atomicAdd(&s_near[b - near], tb);
                    else atomicAdd(&cnt[b], (unsigned long long)tb);
                }
                acc_a += tb;
            }
            const unsigned long long found = wave_sum((unsigned long long)acc_a);
            if (lane == 0 && found) atomicAdd(&cnt[a], found);
            acc_total += found;
            tc_lds_sync();
        }
    }
    flush();
    if (lane == 0 && acc_total) atomicAdd(&s_total, acc_total);
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < kTcNear; k += kTcCoreThreads)
        slab[(uint64_t)blockIdx.x * kTcNear + k] = s_near[k];
    if (threadIdx.x == 0 && s_total) atomicAdd(total, s_total);
}

// cnt[near + k] += the workgroups' credits (the only writer at this point of the stream).
__global__ void tc_core_sum(const uint32_t *__restrict__ slab, uint32_t nwg, uint32_t near, uint32_t n,
                            unsigned long long *cnt) {
    __shared__ unsigned long long s_part[4][kWave];
    const uint32_t lane = threadIdx.x & (kWave - 1), part = threadIdx.x / kWave;
    const uint32_t k = blockIdx.x * kWave + lane;
    unsigned long long c = 0;
    for (uint32_t g = part; g < nwg; g += 4) c += slab[(uint64_t)g * kTcNear + k];
    s_part[part][lane] = c;
    __syncthreads();
    if (part == 0 && near + k < n) {
        c = s_part[0][lane] + s_part[1][lane] + s_part[2][lane] + s_part[3][lane];
        if (c) cnt[near + k] += c;
    }
}

__global__ void tc_to_u32(const unsigned long long *cnt, uint32_t n, uint32_t *out, uint32_t *overflow) {
    uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t v = blockIdx.x * blockDim.x + threadIdx.x; v < n; v += stride) {
        unsigned long long c = cnt[v];
        if (c > 0xffffffffull) atomicOr(overflow, 1u);
        out[v] = (uint32_t)c;
    }
}

template <typename C>
static void tc_prep_layout(C &c, uint64_t E, uint32_t N, uint32_t **deg, uint64_t **vkeys, uint64_t **ekeys,
                           uint32_t **flags, uint32_t **pos, uint32_t **err, void **sw, size_t *swb) {
    int idb = bits_for(N ? N - 1 : 0);
    if (idb == 0) idb = 1;
    *deg = c.template take<uint32_t>(N + 1);
    *vkeys = c.template take<uint64_t>(N + 1);
    *ekeys = c.template take<uint64_t>(E + 1);
    *flags = c.template take<uint32_t>(E + 1);
    *pos = c.template take<uint32_t>(E + 2);
    *err = c.template take<uint32_t>(1);
    size_t s = sort_workspace_bytes(std::max<uint64_t>(E, N), 64, false);
    s = std::max(s, scan_workspace(std::max<uint64_t>(E, N) + 1));
    *sw = c.template take<char>(s);
    *swb = s;
}

// deg[v] += in + out degree of v without self-loops (deg zeroed by the caller),
// from runs of equal ids: the src passes order the keys by src, the dst passes
// by dst.  vkeys (N+1 entries) serves as scratch of the runs' ends, ekeys and sw
// as the sort buffers.
static int tc_degree_counts(const uint32_t *src, const uint32_t *dst, uint64_t E, uint32_t N, uint32_t *deg,
                            uint32_t *err, uint64_t *vkeys, uint64_t *ekeys, void *sw, size_t swb, hipStream_t s) {
    if (!E) return GCHI_OK;
    const int fb = bits_for(N);  // wide enough for n, the skip mark
    const int sb = (fb + 7) / 8 * 8;
    const uint32_t fmask = fb >= 32 ? 0xffffffffu : ((1u << fb) - 1u);
    uint32_t *run_start = reinterpret_cast<uint32_t *>(vkeys), *run_end = run_start + N;
    hipLaunchKernelGGL(tc_degree_pack, dim3(grid_for(E, 256, 65536)), dim3(256), 0, s, src, dst, E, N, sb, ekeys, err);
    GCHI_LAUNCH_CHECK();
    uint64_t *by_dst = nullptr;
    auto by_src = [&](uint64_t *k) { return count_field_runs(k, E, 0, fmask, N, run_start, deg, s, run_end); };
    GCHI_TRY(radix_sort_pairs(PairIO{}, ekeys, nullptr, E, 0, sb, sb + fb, sw, swb, s, &by_dst, err, by_src));
    return count_field_runs(by_dst, E, sb, fmask, N, run_start, deg, s, run_end);
}

}  // namespace gchi

using namespace gchi;

extern "C" int gchi_tc_prepare_workspace(uint64_t nedges, uint32_t nvertices, size_t *bytes) {
    GCHI_CHECK(bytes, GCHI_ERR_INVALID, "null bytes");
    SizerAdapter a;
    uint32_t *d, *f, *p, *e;
    uint64_t *vk, *ek;
    void *sw;
    size_t swb;
    tc_prep_layout(a, nedges, nvertices, &d, &vk, &ek, &f, &p, &e, &sw, &swb);
    *bytes = a.z.off;
    return GCHI_OK;
}

extern "C" int gchi_tc_prepare(const uint32_t *d_src, const uint32_t *d_dst, uint64_t nedges, uint32_t nvertices,
                               uint32_t *d_vertexmap, uint32_t *d_off, uint32_t *d_adj, uint64_t *h_noriented,
                               void *d_work, size_t work_bytes, void *stream) {
    GCHI_CHECK(d_vertexmap && d_off && d_adj && h_noriented && nvertices > 0, GCHI_ERR_INVALID,
               "tc_prepare: null argument");
    GCHI_CHECK(nedges == 0 || (d_src && d_dst), GCHI_ERR_INVALID, "tc_prepare: null edges");
    GCHI_CHECK(nedges < (1ull << 31), GCHI_ERR_UNSUPPORTED, "tc_prepare: E must be < 2^31");
    hipStream_t s = as_stream(stream);
    Carver c(d_work, work_bytes);
    uint32_t *deg, *flags, *pos, *err;
    uint64_t *vkeys, *ekeys;
    void *sw;
    size_t swb;
    tc_prep_layout(c, nedges, nvertices, &deg, &vkeys, &ekeys, &flags, &pos, &err, &sw, &swb);
    GCHI_CHECK(c.ok(), GCHI_ERR_WORKSPACE, "tc_prepare: workspace too small");
    const uint32_t N = nvertices;
    const uint64_t E = nedges;
    int idb = bits_for(N - 1);
    if (idb == 0) idb = 1;
    const int degb = bits_for(2 * E);
    GCHI_CHECK(idb + degb <= 64, GCHI_ERR_UNSUPPORTED, "tc_prepare: degree/id keys exceed 64 bits");
    launch_fill_u32(deg, 0u, N, s);
    launch_fill_u32(err, 0u, 1, s);
    GCHI_TRY(tc_degree_counts(d_src, d_dst, E, N, deg, err, vkeys, ekeys, sw, swb, s));
    hipLaunchKernelGGL(tc_degree_keys, dim3(grid_for(N, 256, 65536)), dim3(256), 0, s, deg, N, idb, vkeys);
    GCHI_LAUNCH_CHECK();
    GCHI_TRY(radix_sort_u64_bits(vkeys, nullptr, nullptr, N, idb, idb + degb, sw, swb, s, nullptr, err));
    hipLaunchKernelGGL(tc_vertexmap, dim3(grid_for(N, 256, 65536)), dim3(256), 0, s, vkeys, N, idb, d_vertexmap);
    const uint64_t sentinel = (2 * idb >= 64) ? ~0ull : ((1ull << (2 * idb)) - 1ull);
    uint32_t *lo_count = deg;  // reuse: degrees are no longer needed
    launch_fill_u32(lo_count, 0u, N + 1, s);
    if (E) {
        hipLaunchKernelGGL(tc_orient_keys, dim3(grid_for(E, 256, 65536)), dim3(256), 0, s, d_src, d_dst, E, N,
                           d_vertexmap, idb, sentinel, ekeys);
        GCHI_LAUNCH_CHECK();
        GCHI_TRY(radix_sort_u64(ekeys, nullptr, E, 2 * idb, sw, swb, s, err));
        hipLaunchKernelGGL(tc_unique_flags, dim3(grid_for(E, 256, 65536)), dim3(256), 0, s, ekeys, E, sentinel,
                           flags);
        GCHI_LAUNCH_CHECK();
        GCHI_TRY(exclusive_scan_u32(flags, pos, E, sw, swb, s));
        uint32_t *lo_start = reinterpret_cast<uint32_t *>(vkeys);  // vertexmap is built: vkeys is free
        hipLaunchKernelGGL(tc_lo_run_starts, dim3(grid_for(E, 256, 65536)), dim3(256), 0, s, ekeys, pos, E, idb,
                           sentinel, N, lo_start);
        hipLaunchKernelGGL(tc_scatter_unique, dim3(grid_for(E, 256, 65536)), dim3(256), 0, s, ekeys, flags, pos, E,
                           idb, sentinel, N, lo_start, d_adj, lo_count);
        GCHI_LAUNCH_CHECK();
    }
    GCHI_TRY(exclusive_scan_u32(lo_count, d_off, N, sw, swb, s));
    uint32_t h_err = 0, h_m = 0;
    GCHI_HIP(hipMemcpyAsync(&h_err, err, 4, hipMemcpyDeviceToHost, s));
    GCHI_HIP(hipMemcpyAsync(&h_m, d_off + N, 4, hipMemcpyDeviceToHost, s));
    GCHI_HIP(hipStreamSynchronize(s));
    GCHI_CHECK(!(h_err & GCHI_WORK_TIMEOUT), GCHI_ERR_TIMEOUT, "tc_prepare: a sort look-back wait gave up");
    GCHI_CHECK(h_err == 0, GCHI_ERR_INVALID, "tc_prepare: vertex id >= nvertices");
    *h_noriented = h_m;
    return GCHI_OK;
}

namespace gchi {

// Scratch of one count.  rows = 0: no core kernel (only cnt and tot are there).
struct TcCount {
    unsigned long long *cnt, *tot;  // [n + 1], [1]
    uint32_t *end, *slab;
    uint2 *maps;
    uint32_t rows, nwg;
};

static int tc_ncu() {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0)
        return v;
    return 256;
}

// The counting launches (the counters are cleared here first).
static int tc_count_impl(const uint32_t *d_off, const uint32_t *d_adj, uint32_t nvertices, uint32_t *d_per_vertex,
                         uint64_t *d_total, uint32_t *d_overflow, const TcCount &w, hipStream_t s) {
    const uint32_t n = nvertices;
    launch_fill_u64(reinterpret_cast<uint64_t *>(w.cnt), 0ull, n, s);
    launch_fill_u64(reinterpret_cast<uint64_t *>(w.tot), 0ull, 1, s);
    launch_fill_u32(d_overflow, 0u, 1, s);
    const int ncu = tc_ncu();
    const uint32_t *end = d_off + 1;
    if (w.rows) {
        const uint32_t base = n > kTcCore ? n - kTcCore : 0u, near = n > kTcNear ? n - kTcNear : 0u;
        const uint32_t first = n - w.rows;
        hipLaunchKernelGGL(tc_core_split, dim3(grid_for(n, 256, 65536)), dim3(256), 0, s, d_off, d_adj, n, base, w.end);
        hipLaunchKernelGGL(tc_core_maps, dim3(grid_for(w.rows, 4, 8192)), dim3(256), 0, s, d_off, d_adj, w.end, first,
                           w.rows, base, w.maps);
        hipLaunchKernelGGL(tc_count_core_kernel, dim3(w.nwg), dim3(kTcCoreThreads), 0, s, d_off, d_adj, w.end, n, base,
                           near, first, w.maps, w.cnt, w.tot, w.slab);
        hipLaunchKernelGGL(tc_core_sum, dim3(kTcNear / kWave), dim3(256), 0, s, w.slab, w.nwg, near, n, w.cnt);
        end = w.end;
    }
    if (!w.rows || n > kTcCore) {
        const uint32_t tail_max = w.rows ? kTcTailMax : kTcTailMaxWhole;
        hipLaunchKernelGGL(tc_count_tail_kernel, dim3(ncu * 6), dim3(kTcTailWaves * kWave), 0, s, d_off, end, d_adj, n,
                           tail_max, w.cnt, w.tot);
        hipLaunchKernelGGL(tc_count_hash_kernel, dim3(grid_for(n, kTcHashWaves, ncu * kTcHashGrid)),
                           dim3(kTcHashWaves * kWave), 0, s, d_off, end, d_adj, n, tail_max, w.cnt, w.tot);
        hipLaunchKernelGGL(tc_count_kernel, dim3(ncu * 8), dim3(kTcWaves * kWave), 0, s, d_off, end, d_adj, n,
                           kTcHashMax, w.cnt, w.tot);
    }
    hipLaunchKernelGGL(tc_to_u32, dim3(grid_for(n, 256, 65536)), dim3(256), 0, s, w.cnt, n, d_per_vertex, d_overflow);
    GCHI_HIP(hipMemcpyAsync(d_total, w.tot, 8, hipMemcpyDeviceToDevice, s));
    GCHI_LAUNCH_CHECK();
    return GCHI_OK;
}

template <typename C>
static void tc_count_layout(C &c, uint32_t nvertices, TcCount *w) {
    w->cnt = c.template take<unsigned long long>((size_t)nvertices + 1);
    w->tot = c.template take<unsigned long long>(1);
    w->rows = 0;
}

// The core kernel's scratch after it: bitmaps for the highest n / 8 ranks (at
// least 16384, at most kTcMapRows: rows of more than kTcList core entries are
// among them in a skewed graph, 64 bytes per vertex), and two workgroups per CU,
// fewer for small graphs, each 64 KB of credits to clear, store and add up: one per
// 32 vertices, at most four to a wavefront (per 64 / 32 / 16 vertices: a clique of
// 100 204 / 115 / 91 us, of 150 231 / 152 / 111; 5,000 vertices with 50,000 random
// edges 105 / 100 / 113).
template <typename C>
static void tc_core_layout(C &c, uint32_t nvertices, TcCount *w) {
    w->rows = std::min(nvertices, std::min(kTcMapRows, std::max(nvertices / 8, kTcNear)));
    w->nwg = std::min<uint32_t>(2 * 256, std::max(1u, nvertices / 32));
    w->end = c.template take<uint32_t>(nvertices);
    w->slab = c.template take<uint32_t>((size_t)w->nwg * kTcNear);
    w->maps = c.template take<uint2>((size_t)w->rows * kWave);
}

// ---- allocation-free counting: scratch in a file-scope device array ----
// Counters for up to GCHI_TC_NOALLOC_MAX_VERTICES vertices, laid out as
// tc_count_layout carves them (256-byte aligned pieces).
constexpr size_t kTcScratchCounts = (((size_t)GCHI_TC_NOALLOC_MAX_VERTICES + 1) * 8 + 255) / 256 * 256;
constexpr size_t kTcScratchBytes = kTcScratchCounts + 256;
static __device__ __align__(256) unsigned char scratch[kTcScratchBytes];

// Device address of each device's copy of scratch (the array's name in host
// code is not a device address), taken once per device with that device
// current.
constexpr int kTcMaxDevices = 64;
static void *g_scratch_ptr[kTcMaxDevices];
static std::mutex g_scratch_mu;

int tc_scratch_setup(int dev) {
    GCHI_CHECK(dev >= 0 && dev < kTcMaxDevices, GCHI_ERR_UNSUPPORTED, "tc scratch: device index >= 64");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (g_scratch_ptr[dev]) return GCHI_OK;
    void *ptr = nullptr;
    GCHI_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    GCHI_CHECK(ptr, GCHI_ERR_HIP, "tc scratch: hipGetSymbolAddress returned null");
    g_scratch_ptr[dev] = ptr;
    return GCHI_OK;
}

}  // namespace gchi

using namespace gchi;

extern "C" int gchi_tc_count_workspace(uint32_t nvertices, size_t *bytes) {
    GCHI_CHECK(bytes, GCHI_ERR_INVALID, "null bytes");
    SizerAdapter a;
    TcCount w;
    tc_count_layout(a, nvertices, &w);
    tc_core_layout(a, nvertices, &w);
    *bytes = a.z.off;
    return GCHI_OK;
}

extern "C" int gchi_tc_count(const uint32_t *d_off, const uint32_t *d_adj, uint32_t nvertices,
                             uint32_t *d_per_vertex, uint64_t *d_total, uint32_t *d_overflow, void *d_work,
                             size_t work_bytes, void *stream) {
    GCHI_CHECK(d_off && d_adj && d_per_vertex && d_total && d_overflow && nvertices > 0, GCHI_ERR_INVALID,
               "tc_count: null argument");
    size_t need = 0;
    gchi_tc_count_workspace(nvertices, &need);
    GCHI_CHECK(d_work && work_bytes >= need, GCHI_ERR_WORKSPACE, "tc_count: workspace too small");
    Carver c(d_work, work_bytes);
    TcCount w;
    tc_count_layout(c, nvertices, &w);
    tc_core_layout(c, nvertices, &w);
    return tc_count_impl(d_off, d_adj, nvertices, d_per_vertex, d_total, d_overflow, w, as_stream(stream));
}

extern "C" int gchi_tc_count_noalloc(const uint32_t *d_off, const uint32_t *d_adj, uint32_t nvertices,
                                     uint32_t *d_per_vertex, uint64_t *d_total, uint32_t *d_overflow, void *stream) {
    GCHI_CHECK(d_off && d_adj && d_per_vertex && d_total && d_overflow && nvertices > 0, GCHI_ERR_INVALID,
               "tc_count_noalloc: null argument");
    GCHI_CHECK(nvertices <= GCHI_TC_NOALLOC_MAX_VERTICES, GCHI_ERR_INVALID,
               "tc_count_noalloc: nvertices exceeds GCHI_TC_NOALLOC_MAX_VERTICES (4,194,304); use gchi_tc_count "
               "with a workspace");
    int dev = 0;
    GCHI_HIP(hipGetDevice(&dev));
    GCHI_TRY(tc_scratch_setup(dev));
    Carver c(g_scratch_ptr[dev], kTcScratchBytes);
    TcCount w;
    tc_count_layout(c, nvertices, &w);  // no bitmaps: the tail and search kernels alone
    GCHI_CHECK(c.ok(), GCHI_ERR_INVALID, "tc_count_noalloc: scratch layout exceeds its array");
    return tc_count_impl(d_off, d_adj, nvertices, d_per_vertex, d_total, d_overflow, w, as_stream(stream));
}

__global__ void relabel_kernel(const uint32_t *src, const uint32_t *dst, uint64_t e, uint32_t n, const uint32_t *map,
                               uint32_t *so, uint32_t *dout, uint32_t *err) {
    uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < e; i += stride) {
        uint32_t s = src[i], d = dst[i];
        if (s >= n || d >= n) {
            atomicOr(err, 1u);
            so[i] = dout[i] = 0;
            continue;
        }
        so[i] = map[s];
        dout[i] = map[d];
    }
}

extern "C" int gchi_degree_order_workspace(uint64_t nedges, uint32_t nvertices, size_t *bytes) {
    return gchi_tc_prepare_workspace(nedges, nvertices, bytes);
}

// order_by_degree's translation table only (orderbydegree.hpp:64-100)
extern "C" int gchi_degree_order(const uint32_t *d_src, const uint32_t *d_dst, uint64_t nedges, uint32_t nvertices,
                                 uint32_t *d_vertexmap, void *d_work, size_t work_bytes, void *stream) {
    GCHI_CHECK(d_vertexmap && nvertices > 0, GCHI_ERR_INVALID, "degree_order: null argument");
    GCHI_CHECK(nedges == 0 || (d_src && d_dst), GCHI_ERR_INVALID, "degree_order: null edges");
    GCHI_CHECK(nedges < (1ull << 31), GCHI_ERR_UNSUPPORTED, "degree_order: E must be < 2^31");
    hipStream_t s = as_stream(stream);
    Carver c(d_work, work_bytes);
    uint32_t *deg, *flags, *pos, *err;
    uint64_t *vkeys, *ekeys;
    void *sw;
    size_t swb;
    tc_prep_layout(c, nedges, nvertices, &deg, &vkeys, &ekeys, &flags, &pos, &err, &sw, &swb);
    GCHI_CHECK(c.ok(), GCHI_ERR_WORKSPACE, "degree_order: workspace too small");
    const uint32_t N = nvertices;
    int idb = bits_for(N - 1);
    if (idb == 0) idb = 1;
    const int degb = bits_for(2 * nedges);
    launch_fill_u32(deg, 0u, N, s);
    launch_fill_u32(err, 0u, 1, s);
    GCHI_TRY(tc_degree_counts(d_src, d_dst, nedges, N, deg, err, vkeys, ekeys, sw, swb, s));
    hipLaunchKernelGGL(tc_degree_keys, dim3(grid_for(N, 256, 65536)), dim3(256), 0, s, deg, N, idb, vkeys);
    GCHI_LAUNCH_CHECK();
    GCHI_TRY(radix_sort_u64_bits(vkeys, nullptr, nullptr, N, idb, idb + degb, sw, swb, s, nullptr, err));
    hipLaunchKernelGGL(tc_vertexmap, dim3(grid_for(N, 256, 65536)), dim3(256), 0, s, vkeys, N, idb, d_vertexmap);
    uint32_t h_err = 0;
    GCHI_HIP(hipMemcpyAsync(&h_err, err, 4, hipMemcpyDeviceToHost, s));
    GCHI_HIP(hipStreamSynchronize(s));
    GCHI_CHECK(!(h_err & GCHI_WORK_TIMEOUT), GCHI_ERR_TIMEOUT, "degree_order: a sort look-back wait gave up");
    GCHI_CHECK(h_err == 0, GCHI_ERR_INVALID, "degree_order: vertex id >= nvertices");
    return GCHI_OK;
}

extern "C" int gchi_relabel_edges(const uint32_t *d_src, const uint32_t *d_dst, uint64_t nedges, uint32_t nvertices,
                                  const uint32_t *d_map, uint32_t *d_src_out, uint32_t *d_dst_out, void *stream) {
    GCHI_CHECK(d_map && (nedges == 0 || (d_src && d_dst && d_src_out && d_dst_out)), GCHI_ERR_INVALID,
               "relabel_edges: null argument");
    if (!nedges) return GCHI_OK;
    hipStream_t s = as_stream(stream);
    uint32_t *err = nullptr;
    GCHI_HIP(device_alloc(&err, 4));
    launch_fill_u32(err, 0u, 1, s);
    hipLaunchKernelGGL(relabel_kernel, dim3(grid_for(nedges, 256, 65536)), dim3(256), 0, s, d_src, d_dst, nedges,
                       nvertices, d_map, d_src_out, d_dst_out, err);
    uint32_t h = 0;
    hipError_t e = hipMemcpyAsync(&h, err, 4, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    (void)hipFree(err);
    if (e != hipSuccess) return hip_fail(e, "relabel_edges", __FILE__, __LINE__);
    GCHI_CHECK(h == 0, GCHI_ERR_INVALID, "relabel_edges: vertex id >= nvertices");
    return GCHI_OK;
}
