// Device decode of a shard's adjacency stream (the bytes of a .adj file).
//
// Reference: memory_shard::load_vertices (src/shards/memoryshard.hpp:448-497)
// parses the stream record by record: a 0 byte and the byte nz after it skip
// 1 + nz vertices; a count byte c (0xff: a uint32 count follows) is followed by
// c uint32 dst ids of the current vertex, which then advances by one.  The
// records have no markers, so where one starts depends on every record before
// it.  Device form, for a stream of n bytes cut into 16 KB chunks:
//   1. sd_exits: every byte position p of a chunk is taken as if a record
//      started there; one workgroup per chunk finds in LDS where the chain from
//      each p leaves the chunk (X).  Sub-blocks of 64 bytes are resolved
//      backwards by one thread each, then merged pairwise.
//   2. sd_supers: a superchunk is K chunks.  A chain enters it within its first
//      1025 bytes (a record of a one-byte count is at most 1017 bytes long) or
//      behind a record of a four-byte count that sd_exits saw crossing into it
//      (the far list); one lane per such entry walks the K tables.
//   3. sd_chain: one wavefront per stream walks the superchunks from position 0,
//      one table entry each, and checks that the chain ends exactly at n;
//      sd_expand then walks the chunks inside every superchunk.
//   4. sd_count / sd_emit: a chunk whose entry is known finds the entries of its
//      256-byte blocks, and one lane per block parses the block's records:
//      counts (edges and vertex advance, scanned into bases), then (src, dst)
//      pairs, through per-edge (byte position, src) words in LDS so that the
//      workgroup writes them out side by side.  The words of a record past the
//      chunk's window go to sd_long in items of 2048.
// The output is the same edge sequence as the reference's parse: the shard's
// edges in stream order, src ids counted from 0.  Several streams (a graph's
// shards) go through one set of launches: a stream table maps every global
// chunk to its stream, and the edges land back to back in stream order.
//
// Bound: vector instructions and LDS in step 1, LDS latency in 4, dependent
// loads in 2 and 3.  Four streams of a scale-21 R-MAT graph (140 MB, 33.6M
// edges): sd_exits 312 us, supers 43, chain 19, expand 49, count 258, emit 149,
// long 34.  The form before it, 3.2 ms: pointer jumping over 32 KB with two
// 32-bit tables of every position written out (1155 us), one thread per stream
// over all chunks (589 us), one thread per 8 KB piece for the counts (463 us) and
// for a queue of records that a binary search per edge expanded (996 us).
#include "common.hpp"
#include "internal.hpp"

namespace gchi {

constexpr int kSdLogChunk = 14;
constexpr uint32_t kSdChunk = 1u << kSdLogChunk;  // bytes per chunk
constexpr int kSdLogBlock = 8;
constexpr uint32_t kSdBlock = 1u << kSdLogBlock;  // bytes per block (one lane's records in sd_count)
constexpr uint32_t kSdBlocks = kSdChunk / kSdBlock;
static_assert(kSdBlocks == kWave, "one wavefront walks a chunk's blocks");
constexpr uint32_t kSdAhead = 1024;   // bytes past the chunk that sd_emit keeps; a one-byte count's record ends
                                      // at most 1016 bytes past its chunk
constexpr uint32_t kSdNear = kSdAhead + 1;  // entries that every superchunk has a table entry for
constexpr uint32_t kSdFar = 256;      // far entries kept per superchunk (others are walked chunk by chunk)
constexpr int kSdThreads = 256;
static_assert(kSdThreads * 64 == kSdChunk, "one thread per 64-byte sub-block");
constexpr uint32_t kSdNone = 0xffffffffu;
constexpr uint32_t kSdNone16 = 0xffffu;
constexpr uint32_t kSdItem = 2048;       // words per sd_long item
constexpr uint32_t kSdWide = 32;         // records of more words are spread over a wavefront

// The streams of one call: stream s has n[s] bytes at adj[s]; its chunks are
// global chunks [cbase[s], cbase[s+1]), its superchunks (of K chunks)
// [sbase[s], sbase[s+1]).
struct SdStreams {
    const uint64_t *adj, *n;
    const uint32_t *cbase, *sbase;
    uint32_t count;
    int lk;  // K = 2^lk
};

GCHI_DEV uint32_t sd_stream_of(const uint32_t *base, uint32_t count, uint32_t g) {  // largest s with base[s] <= g
    uint32_t lo = 0, hi = count - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (base[mid] <= g) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

GCHI_DEV const uint8_t *sd_bytes(const SdStreams &t, uint32_t sid) {
    return reinterpret_cast<const uint8_t *>((uintptr_t)t.adj[sid]);
}

// ---- a chunk in LDS ----
// Bytes and exits carry one word of padding per 64 bytes, so that threads at
// the same place of neighbouring sub-blocks meet different banks.  An exit is
// kept as the byte offset of its own entry in the exit array, so that following
// a chain is a compare and a load; offsets past the chunk's end name positions
// of the chunks behind.  An exit further than kSdReach is a code: kSdCode | r,
// leaving by the four-byte-count record at r, or kSdLost, running past the
// stream's end.
GCHI_DEV uint32_t sd_ba(uint32_t r) { return r + (r >> 6) * 4; }
GCHI_DEV uint32_t sd_enc(uint32_t q) { return 2 * q + (q >> 6) * 4; }
GCHI_DEV uint32_t sd_dec(uint32_t e) { return (e - e / 132 * 4) / 2; }  // 64 entries of 2 bytes and 4 of padding
constexpr uint32_t kSdByteWords = (kSdChunk + 64) / 64 * 17;
constexpr uint32_t kSdByteWordsAhead = (kSdChunk + kSdAhead + 64) / 64 * 17;
constexpr uint32_t kSdExitBytes = kSdChunk / 64 * 132;
constexpr uint32_t kSdReach = kSdChunk + kSdAhead;
constexpr uint32_t kSdCode = 0xc000u;
constexpr uint32_t kSdLost = kSdCode - 1;
static_assert(2 * kSdReach + kSdReach / 64 * 4 < kSdLost && kSdChunk <= 0x4000, "codes lie past every offset");
typedef uint16_t __attribute__((may_alias)) sd_u16;
typedef uint32_t __attribute__((may_alias)) sd_u32;  // two exits
GCHI_DEV uint32_t sd_x(const uint8_t *X, uint32_t e) { return *reinterpret_cast<const sd_u16 *>(X + e); }

GCHI_DEV uint32_t sd_b(const uint32_t *B, uint32_t r) { return reinterpret_cast<const uint8_t *>(B)[sd_ba(r)]; }
GCHI_DEV uint32_t sd_w(const uint32_t *B, uint32_t r) {  // the little-endian word at r
    return sd_b(B, r) | (sd_b(B, r + 1) << 8) | (sd_b(B, r + 2) << 16) | (sd_b(B, r + 3) << 24);
}

// Bytes [start, start + WANT) of the stream, as far as it goes, by the whole
// workgroup; every thread's loads are in flight together.
template <uint32_t WANT>
GCHI_DEV uint32_t sd_load(const uint8_t *__restrict__ adj, uint64_t n, uint64_t start, uint32_t *B) {
    const uint32_t len = n - start < WANT ? (uint32_t)(n - start) : WANT;
    const uint32_t whole = ((uintptr_t)adj & 15u) == 0 ? len / 16 * 16 : 0u;
    constexpr int kLoads = (WANT + kSdThreads * 16 - 1) / (kSdThreads * 16);
    if (whole) {
        uint4 v[kLoads];
#pragma unroll
        for (int k = 0; k < kLoads; k++) {
            const uint32_t i = (k * kSdThreads + threadIdx.x) * 16;
            v[k] = *reinterpret_cast<const uint4 *>(adj + start + (i < whole ? i : 0u));
        }
#pragma unroll
        for (int k = 0; k < kLoads; k++) {
            const uint32_t i = (k * kSdThreads + threadIdx.x) * 16;
            if (i >= whole) continue;
            uint32_t *w = B + sd_ba(i) / 4;
            w[0] = v[k].x;
            w[1] = v[k].y;
            w[2] = v[k].z;
            w[3] = v[k].w;
        }
    }
    for (uint32_t i = whole + threadIdx.x; i < len; i += kSdThreads)
        reinterpret_cast<uint8_t *>(B)[sd_ba(i)] = adj[start + i];
    return len;
}

// The exit of every position r from its 64-byte sub-block (cut at clen): the
// first position at or past its end that the chain from r reaches.  One thread
// per sub-block, from its end backwards, four positions a step: their successors
// lie past the step, except that a zero record of the first two leads to the
// last two.  left = the stream's bytes from the chunk's start; END: fewer than
// kSdReach of them, so that short records can run past the stream too.  far(e)
// sees the end (relative to the chunk) of every four-byte-count record that
// ends past kSdReach.  Bound by its vector instructions (about 15 per position:
// the count of a look-alike 0xff byte comes from the words in registers, and
// only a plausible one takes the branch).
template <bool END, typename F>
GCHI_DEV void sd_subblocks(const uint32_t *B, uint8_t *X, uint32_t clen, uint64_t left, F far) {
    const uint32_t base = threadIdx.x * 64;
    const uint32_t lim = sd_enc(min(clen, base + 64));
    const uint32_t row = threadIdx.x * 17;
    const uint32_t cmax = (uint32_t)min<uint64_t>(left >> 2, 0x3fffffffull);
    // the words of the step, behind it, and the next step's (read ahead of the step's writes)
    uint32_t w1 = B[row + 17], w = B[row + 15];  // row + 16 is padding
#pragma unroll 2
    for (int g = 15; g >= 0; g--) {
        const uint32_t r0 = base + 4 * (uint32_t)g;
        const uint32_t ahead = B[row + (uint32_t)max(g - 1, 0)];
        if (!END || r0 < clen) {
            const uint32_t cnt[4] = {__builtin_amdgcn_alignbyte(w1, w, 1), __builtin_amdgcn_alignbyte(w1, w, 2),
                                     __builtin_amdgcn_alignbyte(w1, w, 3), w1};
            uint32_t q[4], x[4];
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t b = (w >> (8 * j)) & 0xffu, r = r0 + (uint32_t)j;
                const uint32_t p = r + 1 + max(4 * b, 1u);
                q[j] = b == 0xff || (END && p > left) ? kSdLost : sd_enc(p);
                if (b == 0xff && cnt[j] <= cmax) {
                    const uint64_t e = r + 5 + 4ull * cnt[j];
                    if (e <= left && r < clen) {
                        q[j] = e <= kSdReach ? sd_enc((uint32_t)e) : kSdCode | r;
                        if (e > kSdReach) far(e);
                    }
                }
            }
            const uint32_t e0 = 2 * r0 + threadIdx.x * 4;  // sd_enc(r0)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                x[j] = q[j];
                if (q[j] < lim) x[j] = sd_x(X, q[j]);  // of the step itself: replaced below
            }
            x[1] = q[1] == e0 + 6 && q[1] < lim ? x[3] : x[1];
            x[0] = q[0] == e0 + 4 && q[0] < lim ? x[2] : x[0];
            sd_u32 *o = reinterpret_cast<sd_u32 *>(X + e0);
            o[0] = x[0] | (x[1] << 16);
            o[1] = x[2] | (x[3] << 16);
        }
        w1 = w;
        w = ahead;
    }
}

// Blocks of s = 2^ls bytes -> blocks of 2s: the exits of the first halves that
// lie in the second half (which this round does not change) are replaced by
// theirs.  Eight pairs of positions per thread are read, then looked up, then
// written, so that a round waits for LDS twice per eight pairs.
GCHI_DEV void sd_merge(uint8_t *X, uint32_t clen, int ls) {
    const uint32_t end = sd_enc(clen);
    for (uint32_t k0 = threadIdx.x; k0 < kSdChunk / 4; k0 += 8 * kSdThreads) {
        uint32_t e[8], v[8], lim[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const uint32_t k = 2 * (k0 + u * kSdThreads);  // pairs: even positions of the first halves
            const uint32_t blk = k >> ls;
            const uint32_t p = (blk << (ls + 1)) + (k & ((1u << ls) - 1u));
            e[u] = sd_enc(p);
            lim[u] = min(end, sd_enc((blk + 1) << (ls + 1)));
            v[u] = *reinterpret_cast<sd_u32 *>(X + e[u]);
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            uint32_t a = v[u] & 0xffffu, b = v[u] >> 16;
            if (a < lim[u]) a = sd_x(X, a);
            if (b < lim[u]) b = sd_x(X, b);
            v[u] = a | (b << 16);
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (e[u] < end) *reinterpret_cast<sd_u32 *>(X + e[u]) = v[u];
    }
}

// One workgroup per global chunk: the chunk's exit table, and the far entries of
// the superchunks behind.
__global__ __launch_bounds__(kSdThreads) void sd_exits(SdStreams t, uint16_t *__restrict__ X,
                                                       uint32_t *__restrict__ fcount, uint32_t *__restrict__ farq) {
    __shared__ uint32_t B[kSdByteWords];
    __shared__ __align__(4) uint8_t L[kSdExitBytes];
    const uint32_t sid = sd_stream_of(t.cbase, t.count, blockIdx.x);
    const uint64_t n = t.n[sid];
    const uint32_t c = blockIdx.x - t.cbase[sid];
    const uint64_t start = (uint64_t)c * kSdChunk, left = n - start;
    const uint32_t len = sd_load<kSdChunk + 8>(sd_bytes(t, sid), n, start, B);
    const uint32_t clen = min(len, kSdChunk);
    const int lspan = t.lk + kSdLogChunk;
    auto far = [&](uint64_t e) {
        const uint64_t q = start + e, sc = q >> lspan;
        if (q >= n || sc <= (c >> t.lk) || (q & ((1ull << lspan) - 1ull)) < kSdNear) return;
        const uint32_t gsc = t.sbase[sid] + (uint32_t)sc;
        const uint32_t i = atomicAdd(&fcount[gsc], 1u);
        if (i < kSdFar) farq[(uint64_t)gsc * kSdFar + i] = (uint32_t)q;
    };
    __syncthreads();
    if (left >= kSdReach) sd_subblocks<false>(B, L, clen, left, far);
    else sd_subblocks<true>(B, L, clen, left, far);
    __syncthreads();
    for (int ls = 6; ls < kSdLogChunk; ls++) {
        sd_merge(L, clen, ls);
        __syncthreads();
    }
    uint4 *out = reinterpret_cast<uint4 *>(X + (uint64_t)blockIdx.x * kSdChunk);
    for (uint32_t i = threadIdx.x; i < (clen + 7) / 8; i += kSdThreads) {
        const sd_u32 *w = reinterpret_cast<const sd_u32 *>(L + sd_enc(8 * i));
        out[i] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

// The chain from pos to the end of its chunk: one table entry.
GCHI_DEV uint32_t sd_hop(const uint8_t *adj, const uint16_t *x, uint32_t pos) {  // x: the stream's first chunk
    const uint32_t c0 = pos / kSdChunk * kSdChunk;
    const uint32_t v = x[pos];
    if (v < kSdLost) return c0 + sd_dec(v);
    if (v == kSdLost) return kSdNone;
    const uint32_t p = c0 + (v & ~kSdCode);  // its end was checked against n
    const uint32_t cnt = (uint32_t)adj[p + 1] | ((uint32_t)adj[p + 2] << 8) | ((uint32_t)adj[p + 3] << 16) |
                         ((uint32_t)adj[p + 4] << 24);
    return p + 5 + 4 * cnt;
}

// S[gsc][i]: where the chain that enters superchunk gsc at entry i (its i-th
// byte, i < kSdNear, or its far entry i - kSdNear) leaves it.
constexpr uint32_t kSdEntries = kSdNear + kSdFar;
constexpr int kSdSuperThreads = 704;
static_assert(2 * kSdSuperThreads >= (int)kSdEntries, "two workgroups per superchunk");
__global__ __launch_bounds__(kSdSuperThreads) void sd_supers(SdStreams t, const uint16_t *__restrict__ X,
                                                             const uint32_t *__restrict__ fcount,
                                                             const uint32_t *__restrict__ farq,
                                                             uint32_t *__restrict__ S) {
    const uint32_t gsc = blockIdx.x, i = blockIdx.y * kSdSuperThreads + threadIdx.x;
    if (i >= kSdNear + min(fcount[gsc], kSdFar)) return;
    const uint32_t sid = sd_stream_of(t.sbase, t.count, gsc);
    const uint64_t n = t.n[sid], start = (uint64_t)(gsc - t.sbase[sid]) << (t.lk + kSdLogChunk);
    const uint32_t end = (uint32_t)min<uint64_t>(n, start + ((uint64_t)kSdChunk << t.lk));
    const uint16_t *x = X + (uint64_t)t.cbase[sid] * kSdChunk;
    uint64_t from = i < kSdNear ? start + i : (uint64_t)farq[(uint64_t)gsc * kSdFar + (i - kSdNear)];
    uint32_t pos = from < end ? (uint32_t)from : kSdNone;
    while (pos < end) pos = sd_hop(sd_bytes(t, sid), x, pos);
    S[(uint64_t)gsc * kSdEntries + i] = pos;
}

// One wavefront per stream: the chain's entry of every superchunk it enters.
// status: [0] a malformed stream.
__global__ __launch_bounds__(kWave) void sd_chain(SdStreams t, const uint16_t *__restrict__ X,
                                                  const uint32_t *__restrict__ fcount,
                                                  const uint32_t *__restrict__ farq, const uint32_t *__restrict__ S,
                                                  uint32_t *__restrict__ sentry, uint32_t *__restrict__ status) {
    const uint32_t sid = blockIdx.x, lane = threadIdx.x;
    const uint64_t n = t.n[sid];
    const int lspan = t.lk + kSdLogChunk;
    const uint16_t *x = X + (uint64_t)t.cbase[sid] * kSdChunk;
    uint32_t pos = 0;
    while (pos < n) {
        const uint32_t sc = (uint32_t)((uint64_t)pos >> lspan), gsc = t.sbase[sid] + sc;
        const uint32_t off = (uint32_t)(pos - ((uint64_t)sc << lspan));
        if (lane == 0) sentry[gsc] = pos;
        uint32_t to = pos;
        if (off < kSdNear) {
            to = S[(uint64_t)gsc * kSdEntries + off];
        } else {
            const uint32_t nf = min(fcount[gsc], kSdFar);
            for (uint32_t i0 = 0; i0 < nf && to == pos; i0 += kWave) {
                const uint32_t i = i0 + lane;
                const uint64_t hit = __ballot(i < nf && farq[(uint64_t)gsc * kSdFar + i] == pos);
                if (hit) to = S[(uint64_t)gsc * kSdEntries + kSdNear + i0 + (uint32_t)__builtin_ctzll(hit)];
            }
            if (to == pos) {  // the far list was full
                const uint32_t end = (uint32_t)min<uint64_t>(n, ((uint64_t)sc + 1) << lspan);
                while (to < end) to = sd_hop(sd_bytes(t, sid), x, to);
            }
        }
        if (to == kSdNone) {
            if (lane == 0) status[0] = 1;
            return;
        }
        pos = to;
    }
}

// Thread per superchunk: the first record start of each of its chunks.
__global__ void sd_expand(SdStreams t, uint32_t nsuper, const uint16_t *__restrict__ X,
                          const uint32_t *__restrict__ sentry, uint32_t *__restrict__ entry) {
    const uint32_t gsc = blockIdx.x * blockDim.x + threadIdx.x;
    if (gsc >= nsuper) return;
    uint32_t pos = sentry[gsc];
    if (pos == kSdNone) return;
    const uint32_t sid = sd_stream_of(t.sbase, t.count, gsc);
    const uint64_t n = t.n[sid], start = (uint64_t)(gsc - t.sbase[sid]) << (t.lk + kSdLogChunk);
    const uint32_t end = (uint32_t)min<uint64_t>(n, start + ((uint64_t)kSdChunk << t.lk));
    const uint16_t *x = X + (uint64_t)t.cbase[sid] * kSdChunk;
    while (pos < end) {
        entry[t.cbase[sid] + pos / kSdChunk] = pos;
        pos = sd_hop(sd_bytes(t, sid), x, pos);
    }
}

// Where the records of one 64-byte sub-block begin: its first record's position
// in the chunk (kSdNone16: none starts here), and the edges and the vertex
// advance of the chunk's records before it.
struct SdSub {
    uint16_t pos, edges;  // only the chunk's last record can have more edges than fit
    uint32_t adv;
};
constexpr uint32_t kSdSubs = kSdChunk / 64;

// Per global chunk: its sub-blocks, and edges and vertex advance of the records
// starting in it.  One lane per 256-byte block walks the block's records.
__global__ __launch_bounds__(kSdThreads) void sd_count(SdStreams t, const uint32_t *__restrict__ entry,
                                                       SdSub *__restrict__ subs, uint32_t *__restrict__ nedge,
                                                       uint32_t *__restrict__ vadv, uint32_t *__restrict__ status) {
    __shared__ uint32_t B[kSdByteWords];
    __shared__ __align__(8) uint8_t L[kSdExitBytes];
    __shared__ uint32_t s_entry[kSdBlocks];
    const uint32_t g = blockIdx.x, e0 = entry[g];
    if (e0 == kSdNone) {  // no record starts here
        if (threadIdx.x == 0) nedge[g] = vadv[g] = 0u;
        return;
    }
    const uint32_t sid = sd_stream_of(t.cbase, t.count, g);
    const uint64_t n = t.n[sid];
    const uint64_t start = (uint64_t)(g - t.cbase[sid]) * kSdChunk, left = n - start;
    const uint32_t len = sd_load<kSdChunk + 8>(sd_bytes(t, sid), n, start, B);
    const uint32_t clen = min(len, kSdChunk);
    if (threadIdx.x < kSdBlocks) s_entry[threadIdx.x] = kSdNone;
    __syncthreads();
    if (left >= kSdReach) sd_subblocks<false>(B, L, clen, left, [](uint64_t) {});
    else sd_subblocks<true>(B, L, clen, left, [](uint64_t) {});
    __syncthreads();
    for (int ls = 6; ls < kSdLogBlock; ls++) {
        sd_merge(L, clen, ls);
        __syncthreads();
    }
    const uint32_t end = sd_enc(clen);
    if (threadIdx.x == 0)
        for (uint32_t p = sd_enc(e0 - (uint32_t)start); p < end; p = sd_x(L, p)) s_entry[p / (132 * kSdBlock / 64)] = p;
    __syncthreads();
    // the exits are no longer needed: their place takes the sub-blocks
    SdSub *sub = reinterpret_cast<SdSub *>(L);
    sub[threadIdx.x] = SdSub{(uint16_t)kSdNone16, 0, 0};
    __syncthreads();
    if (threadIdx.x < kWave) {
        const uint32_t lane = threadIdx.x, p0 = s_entry[lane];
        uint64_t ne = 0;
        uint32_t va = 0, last = kSdNone;
        if (p0 != kSdNone) {
            const uint32_t pe = min(clen, (lane + 1) * kSdBlock);
            uint64_t p = sd_dec(p0);
            while (p < pe) {  // 64-bit: a truncated stream's last record must not wrap the walk around
                const uint32_t r = (uint32_t)p, b = sd_b(B, r), z = sd_b(B, r + 1);
                if ((r >> 6) != last) {
                    last = r >> 6;
                    sub[last] = SdSub{(uint16_t)r, (uint16_t)ne, va};
                }
                if (b == 0) {
                    va += 1 + z;
                    p += 2;
                    continue;
                }
                const uint32_t cnt = b == 0xff ? sd_w(B, r + 1) : b;
                ne += cnt;
                va += 1;
                p += (b == 0xff ? 5u : 1u) + 4ull * cnt;
            }
        }
        uint64_t ie = ne;
        uint32_t iv = va;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const uint64_t ue = __shfl_up(ie, o, kWave);
            const uint32_t uv = __shfl_up(iv, o, kWave);
            if ((int)lane >= o) {
                ie += ue;
                iv += uv;
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < kSdBlock / 64; k++) {
            SdSub &x = sub[lane * (kSdBlock / 64) + k];
            x.edges += (uint16_t)(ie - ne);
            x.adv += iv - va;
        }
        if (lane == kWave - 1) {
            if (ie > 0xffffffffull) status[1] = 1;
            nedge[g] = (uint32_t)ie;
            vadv[g] = iv;
        }
    }
    __syncthreads();
    subs[(uint64_t)g * kSdSubs + threadIdx.x] = sub[threadIdx.x];
}

// tot[2s], tot[2s+1] = edges and vertex advance of stream s; tot[2 count] = all
// edges; tot[2 count + 1] = the two status words.
__global__ void sd_totals(SdStreams t, const uint64_t *__restrict__ ebase, const uint64_t *__restrict__ vbase,
                          const uint32_t *__restrict__ status, uint64_t *__restrict__ tot) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < t.count) {
        tot[2 * (uint64_t)i] = ebase[t.cbase[i + 1]] - ebase[t.cbase[i]];
        tot[2 * (uint64_t)i + 1] = vbase[t.cbase[i + 1]] - vbase[t.cbase[i]];
    } else if (i == t.count) {
        tot[2 * (uint64_t)i] = ebase[t.cbase[t.count]];
        tot[2 * (uint64_t)i + 1] = (uint64_t)status[0] | ((uint64_t)status[1] << 32);
    }
}

struct SdLong {  // words [pos, pos + 4 cnt) of stream sid are edges eoff .. of src
    uint64_t eoff;
    uint32_t pos, sid, src, cnt;
};

// Per global chunk: the (src, dst) pairs of the records starting in it, at
// their global edge positions; src = the vertex advance before the record
// within its stream.  One thread per sub-block walks its records.
__global__ __launch_bounds__(kSdThreads) void sd_emit(SdStreams t, const SdSub *__restrict__ subs,
                                                      const uint32_t *__restrict__ entry,
                                                      const uint64_t *__restrict__ ebase,
                                                      const uint64_t *__restrict__ vbase,
                                                      uint32_t *__restrict__ out_src, uint32_t *__restrict__ out_dst,
                                                      uint32_t *__restrict__ nitems, SdLong *__restrict__ items) {
    constexpr uint32_t kWords = (kSdChunk + kSdAhead) / 4;  // words the window can hold
    constexpr uint32_t kWideMax = (kSdChunk + kSdAhead) / (4 * kSdWide) + 1;
    __shared__ uint32_t B[kSdByteWordsAhead];
    __shared__ uint16_t s_pos[kWords];
    __shared__ uint32_t s_src[kWords];
    __shared__ uint32_t w_k[kWideMax], w_pos[kWideMax], w_src[kWideMax], w_cnt[kWideMax];
    __shared__ uint32_t s_nwide, s_local;
    const uint32_t g = blockIdx.x;
    if (entry[g] == kSdNone) return;
    const SdSub sub = subs[(uint64_t)g * kSdSubs + threadIdx.x];
    const uint32_t sid = sd_stream_of(t.cbase, t.count, g);
    const uint64_t n = t.n[sid];
    const uint64_t start = (uint64_t)(g - t.cbase[sid]) * kSdChunk;
    if (threadIdx.x == 0) s_nwide = s_local = 0;
    const uint32_t wlen = sd_load<kSdChunk + kSdAhead>(sd_bytes(t, sid), n, start, B);
    const uint64_t eb = ebase[g];
    __syncthreads();
    if (sub.pos != kSdNone16) {
        const uint32_t pe = min(min(wlen, kSdChunk), (threadIdx.x + 1) * 64);
        uint32_t e = sub.edges, v = (uint32_t)(vbase[g] - vbase[t.cbase[sid]]) + sub.adv;
        uint64_t p = sub.pos;
        while (p < pe) {
            const uint32_t r = (uint32_t)p, b = sd_b(B, r), z = sd_b(B, r + 1);
            if (b == 0) {
                v += 1 + z;
                p += 2;
                continue;
            }
            const uint32_t cnt = b == 0xff ? sd_w(B, r + 1) : b;
            const uint32_t pos = r + (b == 0xff ? 5u : 1u);
            // words of the window; the others (of the chunk's last record) go to sd_long
            const uint32_t m = min(cnt, pos + 4 <= wlen ? (wlen - pos) / 4 : 0u);
            if (m <= kSdWide) {
                for (uint32_t j = 0; j < m; j++) {
                    s_pos[e + j] = (uint16_t)(pos + 4 * j);
                    s_src[e + j] = v;
                }
            } else {
                const uint32_t i = atomicAdd(&s_nwide, 1u);
                w_k[i] = e;
                w_pos[i] = pos;
                w_src[i] = v;
                w_cnt[i] = m;
            }
            for (uint32_t j = m; j < cnt; j += kSdItem)
                items[atomicAdd(nitems, 1u)] =
                    SdLong{eb + e + j, (uint32_t)(start + pos + 4 * j), sid, v, cnt - j < kSdItem ? cnt - j : kSdItem};
            e += m;
            v += 1;
            p = pos + 4ull * cnt;
        }
        atomicMax(&s_local, e);
    }
    __syncthreads();
    const uint32_t lane = threadIdx.x & (kWave - 1);
    for (uint32_t i = threadIdx.x / kWave; i < s_nwide; i += kSdThreads / kWave)
        for (uint32_t j = lane; j < w_cnt[i]; j += kWave) {
            s_pos[w_k[i] + j] = (uint16_t)(w_pos[i] + 4 * j);
            s_src[w_k[i] + j] = w_src[i];
        }
    __syncthreads();
    const uint32_t local = s_local;
    for (uint32_t k = threadIdx.x; k < local; k += kSdThreads) {
        const uint32_t r = s_pos[k], r4 = r & ~3u;
        const uint32_t lo = B[sd_ba(r4) / 4], hi = B[sd_ba(r4 + 4) / 4];
        out_src[eb + k] = s_src[k];
        out_dst[eb + k] = (uint32_t)((((uint64_t)hi << 32) | lo) >> (8 * (r & 3u)));
    }
}

// One wavefront per item: words of long records past their chunk's window.
__global__ __launch_bounds__(kSdThreads) void sd_long(SdStreams t, const uint32_t *__restrict__ nitems,
                                                      const SdLong *__restrict__ items,
                                                      uint32_t *__restrict__ out_src,
                                                      uint32_t *__restrict__ out_dst) {
    const uint32_t lane = threadIdx.x & (kWave - 1), count = *nitems;
    for (uint32_t i = (blockIdx.x * kSdThreads + threadIdx.x) / kWave; i < count;
         i += gridDim.x * (kSdThreads / kWave)) {
        const SdLong it = items[i];
        const uint8_t *adj = sd_bytes(t, it.sid);
        const uint8_t *p = adj + it.pos;
        const uint32_t sh = (uint32_t)((uintptr_t)p & 3u);
        const uint32_t *w = reinterpret_cast<const uint32_t *>(p - sh);  // it.pos >= 5: not before the stream
        const uint8_t *end = adj + t.n[it.sid];
        for (uint32_t j = lane; j < it.cnt; j += kWave) {
            uint32_t d;
            if (sh == 0) {
                d = w[j];
            } else if (reinterpret_cast<const uint8_t *>(w + j + 2) <= end) {
                d = (uint32_t)((((uint64_t)w[j + 1] << 32) | w[j]) >> (8 * sh));
            } else {  // the stream's last word
                const uint8_t *q = p + 4ull * j;
                d = (uint32_t)q[0] | ((uint32_t)q[1] << 8) | ((uint32_t)q[2] << 16) | ((uint32_t)q[3] << 24);
            }
            out_src[it.eoff + j] = it.src;
            out_dst[it.eoff + j] = d;
        }
    }
}

struct SdShape {
    uint64_t bytes = 0, chunks = 0, supers = 0;
    uint32_t count = 0;
    int lk = 3;
};

// Chunks per superchunk: about the square root of the longest stream's chunks,
// so that the walk inside a superchunk and the walk over them are about equally
// long (both are chains of dependent loads).
static SdShape sd_shape(const uint64_t *h_nbytes, uint32_t count) {
    SdShape z;
    z.count = count;
    uint64_t most = 0;
    for (uint32_t i = 0; i < count; i++) {
        const uint64_t c = div_up(h_nbytes[i], kSdChunk);
        z.bytes += h_nbytes[i];
        z.chunks += c;
        most = std::max(most, c);
    }
    while (z.lk < 9 && (2ull << (2 * z.lk)) < most) z.lk++;
    for (uint32_t i = 0; i < count; i++) z.supers += div_up(div_up(h_nbytes[i], kSdChunk), 1ull << z.lk);
    return z;
}

struct SdWork {
    uint64_t *tables;  // adj[count], n[count], then cbase[count + 1], sbase[count + 1] (u32)
    uint16_t *X;
    SdSub *subs;
    uint32_t *entry, *sentry;             // one fill clears both
    uint32_t *fcount, *status, *nitems;   // one fill clears all three
    uint32_t *farq, *S, *nedge, *vadv;
    SdLong *items;
    uint64_t *ebase, *vbase, *tot;
    void *scan;
    size_t scan_bytes;
};

template <typename C>
static void sd_layout(C &c, const SdShape &z, SdWork *w) {
    const uint64_t nch = z.chunks, ns = z.supers, cnt = z.count;
    auto *tb = c.template take<uint64_t>(3 * cnt + 1);
    auto *X = c.template take<uint16_t>(nch * kSdChunk);
    auto *sub = c.template take<SdSub>(nch * kSdSubs);
    auto *en = c.template take<uint32_t>(nch + ns);
    auto *fc = c.template take<uint32_t>(ns + 3);
    auto *fq = c.template take<uint32_t>(ns * kSdFar);
    auto *S = c.template take<uint32_t>(ns * kSdEntries);
    auto *ne = c.template take<uint32_t>(nch + 1);
    auto *va = c.template take<uint32_t>(nch + 1);
    auto *it = c.template take<SdLong>(z.bytes / 4 / kSdItem + nch + 1);  // a chunk's last record: one item not full
    auto *eb = c.template take<uint64_t>(nch + 1);
    auto *vb = c.template take<uint64_t>(nch + 1);
    auto *to = c.template take<uint64_t>(2 * cnt + 2);
    const size_t sb = scan_workspace((size_t)nch + 1);
    void *sw = c.template take<char>(sb);
    if (w) *w = SdWork{tb, X, sub, en, en + nch, fc, fc + ns, fc + ns + 2, fq, S, ne, va, it, eb, vb, to, sw, sb};
}

}  // namespace gchi

using namespace gchi;

extern "C" int gchi_shard_decode_many_workspace(const uint64_t *h_nbytes, uint32_t nstreams, size_t *bytes) {
    GCHI_CHECK(bytes && (nstreams == 0 || h_nbytes), GCHI_ERR_INVALID, "shard_decode: null argument");
    SizerAdapter a;
    sd_layout(a, sd_shape(h_nbytes, nstreams), nullptr);
    *bytes = a.z.off;
    return GCHI_OK;
}

extern "C" int gchi_shard_decode_workspace(uint64_t nbytes, size_t *bytes) {
    return gchi_shard_decode_many_workspace(&nbytes, 1, bytes);
}

extern "C" int gchi_shard_decode_many(const uint8_t *const *h_adj, const uint64_t *h_nbytes, uint32_t nstreams,
                                      uint32_t *d_src, uint32_t *d_dst, uint64_t max_edges, uint64_t *h_nedges,
                                      uint64_t *h_vend, void *d_work, size_t work_bytes, void *stream) {
    GCHI_CHECK(nstreams == 0 || (h_adj && h_nbytes && h_nedges), GCHI_ERR_INVALID, "shard_decode: null argument");
    GCHI_CHECK((d_src == nullptr) == (d_dst == nullptr), GCHI_ERR_INVALID, "shard_decode: give both outputs or none");
    for (uint32_t i = 0; i < nstreams; i++) {
        GCHI_CHECK(h_nbytes[i] == 0 || h_adj[i], GCHI_ERR_INVALID, "shard_decode: null stream");
        GCHI_CHECK(h_nbytes[i] < 0xffffffffull, GCHI_ERR_UNSUPPORTED, "shard_decode: streams of 4 GiB or more");
        h_nedges[i] = 0;
        if (h_vend) h_vend[i] = 0;
    }
    const SdShape z = sd_shape(h_nbytes, nstreams);
    if (z.chunks == 0) return GCHI_OK;  // no stream holds a byte
    GCHI_CHECK(z.chunks * kSdSubs < 0x7fffffffull, GCHI_ERR_UNSUPPORTED, "shard_decode: too many bytes in one call");
    // the stream tables, uploaded in one copy
    const size_t cnt = nstreams;
    std::vector<uint64_t> tables(3 * cnt + 1, 0);
    uint32_t *t_c = reinterpret_cast<uint32_t *>(tables.data() + 2 * cnt), *t_s = t_c + cnt + 1;
    for (size_t i = 0; i < cnt; i++) {
        const uint64_t nc = div_up(h_nbytes[i], kSdChunk);
        tables[i] = (uint64_t)(uintptr_t)h_adj[i];
        tables[cnt + i] = h_nbytes[i];
        t_c[i + 1] = t_c[i] + (uint32_t)nc;
        t_s[i + 1] = t_s[i] + (uint32_t)div_up(nc, 1ull << z.lk);
    }
    size_t need = 0;
    gchi_shard_decode_many_workspace(h_nbytes, nstreams, &need);
    GCHI_CHECK(d_work && work_bytes >= need, GCHI_ERR_WORKSPACE, "shard_decode: workspace too small");
    hipStream_t s = as_stream(stream);
    Carver c(d_work, work_bytes);
    SdWork w;
    sd_layout(c, z, &w);
    GCHI_HIP(hipMemcpyAsync(w.tables, tables.data(), 8 * tables.size(), hipMemcpyHostToDevice, s));
    const uint32_t *d_c = reinterpret_cast<const uint32_t *>(w.tables + 2 * cnt);
    const SdStreams T{w.tables, w.tables + cnt, d_c, d_c + cnt + 1, nstreams, z.lk};
    const uint32_t nch = (uint32_t)z.chunks, ns = (uint32_t)z.supers;
    const dim3 blk(kSdThreads);
    launch_fill_u32(w.entry, kSdNone, (size_t)nch + ns, s);
    launch_fill_u32(w.fcount, 0u, (size_t)ns + 3, s);
    hipLaunchKernelGGL(sd_exits, dim3(nch), blk, 0, s, T, w.X, w.fcount, w.farq);
    hipLaunchKernelGGL(sd_supers, dim3(ns, 2), dim3(kSdSuperThreads), 0, s, T, w.X, w.fcount, w.farq, w.S);
    hipLaunchKernelGGL(sd_chain, dim3(nstreams), dim3(kWave), 0, s, T, w.X, w.fcount, w.farq, w.S, w.sentry,
                       w.status);
    hipLaunchKernelGGL(sd_expand, dim3((unsigned)div_up(ns, kWave)), dim3(kWave), 0, s, T, ns, w.X, w.sentry, w.entry);
    hipLaunchKernelGGL(sd_count, dim3(nch), blk, 0, s, T, w.entry, w.subs, w.nedge, w.vadv, w.status);
    GCHI_LAUNCH_CHECK();
    GCHI_TRY(exclusive_scan_u32_to_u64(w.nedge, w.ebase, nch, w.scan, w.scan_bytes, s));
    GCHI_TRY(exclusive_scan_u32_to_u64(w.vadv, w.vbase, nch, w.scan, w.scan_bytes, s));
    hipLaunchKernelGGL(sd_totals, dim3((unsigned)div_up(cnt + 1, 256)), dim3(256), 0, s, T, w.ebase, w.vbase,
                       w.status, w.tot);
    GCHI_LAUNCH_CHECK();
    std::vector<uint64_t> tot(2 * cnt + 2);
    GCHI_HIP(hipMemcpyAsync(tot.data(), w.tot, 8 * tot.size(), hipMemcpyDeviceToHost, s));
    GCHI_HIP(hipStreamSynchronize(s));
    const uint64_t st = tot[2 * cnt + 1];
    GCHI_CHECK((uint32_t)st == 0, GCHI_ERR_FORMAT, "shard_decode: truncated stream (a record runs past its end)");
    GCHI_CHECK((st >> 32) == 0, GCHI_ERR_OVERFLOW, "shard_decode: a chunk's edge count exceeds 32 bits");
    for (size_t i = 0; i < cnt; i++) {
        h_nedges[i] = tot[2 * i];
        GCHI_CHECK(tot[2 * i + 1] <= 0x100000000ull, GCHI_ERR_OVERFLOW, "shard_decode: vertex ids exceed 32 bits");
        if (h_vend) h_vend[i] = tot[2 * i + 1];
    }
    if (!d_src) return GCHI_OK;
    GCHI_CHECK(tot[2 * cnt] <= max_edges, GCHI_ERR_INVALID, "shard_decode: the streams hold more than max_edges edges");
    hipLaunchKernelGGL(sd_emit, dim3(nch), blk, 0, s, T, w.subs, w.entry, w.ebase, w.vbase, d_src, d_dst, w.nitems,
                       w.items);
    hipLaunchKernelGGL(sd_long, dim3(1024), blk, 0, s, T, w.nitems, w.items, d_src, d_dst);
    GCHI_LAUNCH_CHECK();
    return GCHI_OK;
}

extern "C" int gchi_shard_decode(const uint8_t *d_adj, uint64_t nbytes, uint32_t *d_src, uint32_t *d_dst,
                                 uint64_t max_edges, uint64_t *h_nedges, uint64_t *h_vend, void *d_work,
                                 size_t work_bytes, void *stream) {
    GCHI_CHECK(h_nedges, GCHI_ERR_INVALID, "shard_decode: null h_nedges");
    return gchi_shard_decode_many(&d_adj, &nbytes, 1, d_src, d_dst, max_edges, h_nedges, h_vend, d_work, work_bytes,
                                  stream);
}
