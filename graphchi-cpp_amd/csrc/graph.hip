// Device graph construction: degree histograms and the in-edge (CSC) view.
//
// The reference keeps every interval's in-edges in its memory shard, sorted by
// src (src/preprocessing/sharder.hpp:640, src/shards/memoryshard.hpp:448-497),
// and per-vertex {indegree, outdegree} in <G>_degs.bin
// (src/engine/auxdata/degree_data.hpp:45-48).  Here the whole graph is one
// resident CSC sorted by (dst, src): in_off[N+1], in_src[E], plus degree arrays.
#include "common.hpp"
#include "internal.hpp"

namespace gchi {

unsigned grid_for(uint64_t n, unsigned threads, unsigned cap) {
    uint64_t b = div_up(n, threads);
    if (b == 0) b = 1;
    if (b > cap) b = cap;
    return (unsigned)b;
}

// Counting by sorted runs.  Device-wide atomics on random counters run at a few
// billion per second on this part whatever the spread of the ids, so the CSC
// build counts degrees from runs of equal ids in sorted keys instead: the key
// is (dst << sb) | src with sb = vb rounded up to a whole 8-bit digit, the
// first sb/8 radix passes leave the keys ordered by src alone (out-degrees are
// the lengths of its runs), and the remaining passes finish the (dst, src)
// order (in-degrees are the lengths of the dst runs).

// One pass over the keys: run_start[f] = index of the first key of the run of
// field f, run_end[f] = one past its last key, each by the one thread that sees
// the field change.  It is bound by the read of the keys, so a thread has
// kRunKeys of them in flight: a pass for the starts and one for the lengths, a
// key at a time, took 190 us on 33.6M 64-bit keys; 69.
constexpr int kRunKeys = 8;
template <typename K>
__global__ __launch_bounds__(256) void field_runs(const K *__restrict__ k, uint64_t n, int shift, uint32_t mask,
                                                  uint32_t nv, uint32_t *__restrict__ run_start,
                                                  uint32_t *__restrict__ run_end) {
    constexpr uint64_t kSpan = 256 * kRunKeys;
    for (uint64_t base = (uint64_t)blockIdx.x * kSpan; base < n; base += (uint64_t)gridDim.x * kSpan) {
        K key[kRunKeys], next[kRunKeys];
#pragma unroll
        for (int u = 0; u < kRunKeys; u++) {
            const uint64_t i = base + (uint64_t)u * 256 + threadIdx.x;
            key[u] = k[i < n ? i : n - 1];
            next[u] = k[i + 1 < n ? i + 1 : n - 1];
        }
#pragma unroll
        for (int u = 0; u < kRunKeys; u++) {
            const uint64_t i = base + (uint64_t)u * 256 + threadIdx.x;
            if (i >= n) continue;
            const uint32_t f = (uint32_t)(key[u] >> shift) & mask, g = (uint32_t)(next[u] >> shift) & mask;
            if (i == 0 && f < nv) run_start[f] = 0;
            if (i + 1 == n || f != g) {
                if (f < nv) run_end[f] = (uint32_t)(i + 1);
                if (i + 1 < n && g < nv) run_start[g] = (uint32_t)(i + 1);
            }
        }
    }
}

// cnt[f] = (or +=, with accumulate) run_end[f] - run_start[f] where a run ended
// (run_end, which may be cnt, is 0 elsewhere)
__global__ void field_run_counts(const uint32_t *run_start, const uint32_t *run_end, uint32_t nv, uint32_t *cnt,
                                 int accumulate) {
    uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t f = blockIdx.x * blockDim.x + threadIdx.x; f < nv; f += stride) {
        const uint32_t e = run_end[f];
        if (!e) continue;
        const uint32_t len = e - run_start[f];
        cnt[f] = accumulate ? cnt[f] + len : len;
    }
}

template <typename K>
int count_field_runs(const K *keys, uint64_t n, int shift, uint32_t mask, uint32_t nv, uint32_t *run_start,
                     uint32_t *cnt, hipStream_t s, uint32_t *run_end) {
    if (n == 0) return GCHI_OK;
    if (run_end) launch_fill_u32(run_end, 0u, nv, s);
    uint32_t *end = run_end ? run_end : cnt;
    hipLaunchKernelGGL(field_runs<K>, dim3(grid_for(div_up(n, kRunKeys), 256, 65536)), dim3(256), 0, s, keys, n,
                       shift, mask, nv, run_start, end);
    hipLaunchKernelGGL(field_run_counts, dim3(grid_for(nv, 256, 65536)), dim3(256), 0, s, run_start, end, nv, cnt,
                       run_end ? 1 : 0);
    GCHI_LAUNCH_CHECK();
    return GCHI_OK;
}

template int count_field_runs<uint32_t>(const uint32_t *, uint64_t, int, uint32_t, uint32_t, uint32_t *, uint32_t *,
                                        hipStream_t, uint32_t *);
template int count_field_runs<uint64_t>(const uint64_t *, uint64_t, int, uint32_t, uint32_t, uint32_t *, uint32_t *,
                                        hipStream_t, uint32_t *);

struct CscBits {
    int vb;  // bits of a vertex id
    int sb;  // bits the src field takes in a key (vb rounded up to 8)
};
static CscBits csc_bits(uint32_t N) {
    int vb = bits_for(N ? N - 1 : 0);
    if (vb == 0) vb = 1;
    return CscBits{vb, (vb + 7) / 8 * 8};
}

template <typename C>
static void csc_layout(C &c, uint64_t E, uint32_t N, uint64_t **keys, uint32_t **indeg, uint32_t **run_start,
                       uint32_t **err, void **sw, size_t *sw_bytes) {
    const CscBits cb = csc_bits(N);
    *err = c.template take<uint32_t>(1);  // status word (GCHI_WORK_* bits) first: gchi_work_status reads it
    *keys = c.template take<uint64_t>(E ? E : 1);
    *indeg = c.template take<uint32_t>(N ? N : 1);
    *run_start = c.template take<uint32_t>(N ? N : 1);
    size_t ss = std::max(sort_workspace_bytes(E, cb.sb + cb.vb, false), scan_workspace((size_t)N + 1));
    *sw = c.template take<char>(ss);
    *sw_bytes = ss;
}

int csc_build(const uint32_t *src, const uint32_t *dst, uint64_t E, uint32_t N, uint32_t *in_off, uint32_t *in_src,
              uint32_t *outdeg, uint32_t *indeg_out, void *work, size_t work_bytes, hipStream_t s) {
    GCHI_CHECK(E <= kMaxEdges, GCHI_ERR_UNSUPPORTED, "csc_build: E must be <= 2^32 - 2^25 (uint32 offsets)");
    GCHI_CHECK(in_off && (E == 0 || (src && dst && in_src)), GCHI_ERR_INVALID, "csc_build: null pointer");
    Carver c(work, work_bytes);
    uint64_t *keys;
    uint32_t *indeg, *run_start, *err;
    void *sw;
    size_t swb;
    csc_layout(c, E, N, &keys, &indeg, &run_start, &err, &sw, &swb);
    GCHI_CHECK(c.ok(), GCHI_ERR_WORKSPACE, "csc_build: workspace too small");
    uint32_t *ind = indeg_out ? indeg_out : indeg;
    const CscBits cb = csc_bits(N);
    const uint32_t vmask = cb.vb >= 32 ? 0xffffffffu : ((1u << cb.vb) - 1u);
    launch_fill_u32(err, 0u, 1, s);
    if (outdeg) launch_fill_u32(outdeg, 0u, N, s);
    launch_fill_u32(ind, 0u, N, s);
    if (E) {
        PairIO io;
        io.lo_in = src;
        io.hi_in = dst;
        io.lo_out = in_src;
        io.id_bits = cb.sb;
        io.limit = N;
        io.lo_mask = vmask;
        // src passes: keys ordered by src; out-degrees from its runs
        auto by_src = [&](uint64_t *k) {
            return outdeg ? count_field_runs(k, E, 0, vmask, N, run_start, outdeg, s) : GCHI_OK;
        };
        // dst passes (stable, so src order within a dst run is kept): the last
        // one stores src to in_src and dst beside it
        uint64_t *by_dst = nullptr;
        GCHI_TRY(radix_sort_pairs(io, keys, nullptr, E, 0, cb.sb, cb.sb + cb.vb, sw, swb, s, &by_dst, err, by_src));
        GCHI_TRY(count_field_runs(reinterpret_cast<const uint32_t *>(by_dst), E, 0, vmask, N, run_start, ind, s));
    }
    GCHI_TRY(exclusive_scan_u32(ind, in_off, N, sw, swb, s));
    return GCHI_OK;
}

size_t csc_workspace(uint64_t E, uint32_t N) {
    SizerAdapter a;
    uint64_t *k;
    uint32_t *i, *r, *e;
    void *sw;
    size_t swb;
    csc_layout(a, E, N, &k, &i, &r, &e, &sw, &swb);
    return a.z.off;
}

}  // namespace gchi

using namespace gchi;

extern "C" int gchi_csc_build_workspace(uint64_t nedges, uint32_t nvertices, size_t *bytes) {
    GCHI_CHECK(bytes, GCHI_ERR_INVALID, "null bytes");
    *bytes = csc_workspace(nedges, nvertices);
    return GCHI_OK;
}

extern "C" int gchi_csc_build(const uint32_t *d_src, const uint32_t *d_dst, uint64_t nedges, uint32_t nvertices,
                              uint32_t *d_in_off, uint32_t *d_in_src, uint32_t *d_outdeg, uint32_t *d_indeg,
                              void *d_work, size_t work_bytes, void *stream) {
    return csc_build(d_src, d_dst, nedges, nvertices, d_in_off, d_in_src, d_outdeg, d_indeg, d_work, work_bytes,
                     as_stream(stream));
}
