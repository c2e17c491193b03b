// Edge-list text parsed on the device: the input path of
// convert_edgelist (src/preprocessing/conversions.hpp:210-288) feeding
// sharder::preprocessing_add_edge (src/preprocessing/sharder.hpp:427-446).
//
// The reference reads the file line by line with fgets (lines of at most 1023
// bytes), drops the trailing newline, skips lines whose first byte is '#' or
// '%', splits the rest with strtok on tab, comma and space, takes from =
// atoi(token 1) and to = atoi(token 2) (a third token is the edge value), stops
// with an assertion when a line has fewer than two tokens, and drops
// self-loops.  Here the text is in HBM and parsed in parallel:
//   * one wavefront per 4 KiB chunk, one lane per 64-byte slice; a line
//     belongs to the slice its first byte lies in (the file start, or the byte
//     after a newline), and that lane parses it to its end (past the slice and
//     the chunk if need be).  The chunk goes through LDS (see parse_pass);
//   * a count pass gives every chunk its number of kept edges, a scan gives
//     its output offset, and a write pass parses again and writes the pairs in
//     file order (lanes in order, lines in order within a lane).
// A line with fewer than two tokens, or of 1023 bytes or more (fgets would
// split it), is an error reported with the byte offset where it starts.
#include "common.hpp"
#include "internal.hpp"

namespace gchi {

constexpr uint32_t kParseChunk = 4096;
constexpr uint32_t kParseSlice = kParseChunk / kWave;  // 64 bytes per lane
constexpr uint32_t kParseMaxLine = 1023;               // fgets(s, 1024, f) reads at most 1023 bytes

GCHI_DEV bool is_delim(uint8_t c) { return c == '\t' || c == ',' || c == ' '; }

// One forward scan of the line at s: get(p) is byte p, for p < lim.  Returns 1
// and the pair for an edge line, 0 for a comment, -1 for a line with fewer than
// two tokens or one too long; -2 when the line goes on past lim < n (end = the
// end of the text) without being decided.  atoi of a token: leading \r, \v, \f,
// a sign, then decimal digits up to the first other byte; the value wraps to
// 32 bits as the reference's int-to-vid_t cast.
template <typename P, typename Get>
GCHI_DEV int parse_line(Get get, P s, P lim, bool lim_is_end, uint32_t &from, uint32_t &to) {
    P p = s;
    auto at = [&](P q) -> uint32_t { return q < lim ? get(q) : (uint32_t)'\n'; };
    uint32_t c = at(p);
    const bool comment = c == '#' || c == '%';
    int tokens = 0;
    if (!comment) {
#pragma unroll 1
        for (; tokens < 2; tokens++) {
            while (is_delim((uint8_t)c)) c = at(++p);
            if (c == '\n') break;
            while (c == '\r' || c == '\v' || c == '\f') c = at(++p);
            bool neg = false;
            if (c == '+' || c == '-') {
                neg = c == '-';
                c = at(++p);
            }
            uint32_t v = 0;
            while (c - '0' <= 9u) {
                v = v * 10u + (c - '0');
                c = at(++p);
            }
            while (c != '\n' && !is_delim((uint8_t)c)) c = at(++p);
            if (neg) v = 0u - v;
            if (tokens == 0) from = v;
            else to = v;
        }
    }
    while (c != '\n') c = at(++p);
    if (p >= lim && !lim_is_end) return -2;
    if ((uint64_t)(p - s) >= kParseMaxLine) return -1;
    return comment ? 0 : (tokens == 2 ? 1 : -1);
}

// The line at s, from global memory: for the lines that the chunk's LDS window
// does not hold whole.
GCHI_DEV int parse_line_global(const uint8_t *t, uint64_t n, uint64_t s, uint32_t &from, uint32_t &to) {
    // one byte more than an accepted line can have decides it
    const uint64_t lim = min(n, s + kParseMaxLine + 1);
    const int r = parse_line<uint64_t>([&](uint64_t q) { return (uint32_t)t[q]; }, s, lim, lim == n, from, to);
    return r == -2 ? -1 : r;
}

// A wavefront's LDS window: its chunk and kParseAhead bytes more, with 4 bytes
// of padding after every 64 so that the lanes, which all scan at about the same
// place of their own slices, meet different banks.
constexpr uint32_t kParseAhead = 128;
constexpr uint32_t kParseWindow = kParseChunk + kParseAhead;
constexpr uint32_t kParseLds = kParseWindow / 64 * 68;
constexpr int kParseWaves = 4;

GCHI_DEV uint32_t parse_addr(uint32_t p) { return p + (p >> 6) * 4; }

GCHI_DEV void parse_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// WRITE = 0: kept edges per chunk and per lane, errors.  WRITE = 1: the pairs at
// the chunk's scanned offset and the lanes' counts, max id.
//
// Bound: byte loads, not bandwidth.  A lane that walks its slice in global
// memory waits for a cache round trip per byte (316 us a pass for 45 MB of text,
// 0.14 TB/s).  Here the wavefront copies its chunk to LDS with 16-byte loads
// (text aligned to 16; byte loads otherwise), each lane turns its slice into a
// bit mask of line starts, and the lines are scanned in LDS (55 us); only
// a line that runs more than kParseAhead bytes past the chunk is scanned in
// global memory.
template <int WRITE>
__global__ __launch_bounds__(kParseWaves *kWave) void parse_pass(const uint8_t *__restrict__ t, uint64_t n,
                                                                 uint64_t nchunks, uint32_t *chunk_cnt,
                                                                 uint8_t *__restrict__ lane_cnt,
                                                                 const uint64_t *__restrict__ chunk_off,
                                                                 uint32_t *__restrict__ src,
                                                                 uint32_t *__restrict__ dst, uint64_t max_edges,
                                                                 unsigned long long *bad_pos, uint32_t *maxid) {
    __shared__ __align__(16) uint8_t s_text[kParseWaves][kParseLds];
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    uint8_t *B = s_text[wave];
    const uint64_t wid = (uint64_t)blockIdx.x * kParseWaves + wave;
    const uint64_t nw = (uint64_t)gridDim.x * kParseWaves;
    const bool aligned = ((uintptr_t)t & 15u) == 0;
    uint32_t top = 0;
    for (uint64_t c = wid; c < nchunks; c += nw) {
        const uint64_t base = c * kParseChunk;
        const uint32_t win = (uint32_t)min<uint64_t>(kParseWindow, n - base);
        const uint32_t whole = aligned ? win / 16 * 16 : 0u;
        for (uint32_t p = (uint32_t)lane * 16; p < whole; p += kWave * 16) {
            const uint4 v = *reinterpret_cast<const uint4 *>(t + base + p);
            uint32_t *w = reinterpret_cast<uint32_t *>(B + parse_addr(p));  // 16 bytes of one 64-byte row
            w[0] = v.x;
            w[1] = v.y;
            w[2] = v.z;
            w[3] = v.w;
        }
        for (uint32_t p = whole + lane; p < win; p += kWave) B[parse_addr(p)] = t[base + p];
        parse_lds_sync();
        // newline bits of the lane's slice, then its line starts
        const uint32_t lo = (uint32_t)lane * kParseSlice;
        const uint32_t len = win > lo ? min(kParseSlice, win - lo) : 0u;
        uint64_t nl = 0;
        const uint32_t *W = reinterpret_cast<const uint32_t *>(B + parse_addr(lo));
#pragma unroll
        for (int k = 0; k < (int)kParseSlice / 4; k++) {
            const uint32_t x = W[k] ^ 0x0a0a0a0au;  // bytes past the text are masked below
            // exact zero-byte test, one bit per byte, gathered to 4 bits
            const uint32_t z = ~(((x & 0x7f7f7f7fu) + 0x7f7f7f7fu) | x | 0x7f7f7f7fu);
            nl |= (uint64_t)(((z >> 7) * 0x10204080u) >> 28) << (4 * k);
        }
        if (len < kParseSlice) nl &= (1ull << len) - 1ull;
        uint32_t before = __shfl_up((uint32_t)(nl >> 63), 1, kWave);
        if (lane == 0) before = base == 0 || t[base - 1] == '\n' ? 1u : 0u;
        uint64_t starts = (nl << 1) | before;
        if (len < kParseSlice) starts &= (1ull << len) - 1ull;

        auto line = [&](uint32_t s, uint32_t &f, uint32_t &to) {
            int r = parse_line<uint32_t>([&](uint32_t q) { return (uint32_t)B[parse_addr(q)]; }, s, win,
                                         base + win == n, f, to);
            if (r == -2) r = parse_line_global(t, n, base + s, f, to);
            return r;
        };
        if (!WRITE) {
            uint32_t kept = 0;  // at most 32: every line takes at least 2 bytes with its newline, edge lines 4
            for (uint64_t m = starts; m; m &= m - 1) {
                const uint32_t s = lo + (uint32_t)__builtin_ctzll(m);
                uint32_t f = 0, to = 0;
                const int r = line(s, f, to);
                if (r < 0) atomicMin(bad_pos, (unsigned long long)(base + s));
                if (r > 0 && f != to) kept++;
            }
            lane_cnt[c * kWave + lane] = (uint8_t)kept;
            const uint32_t tot = wave_sum(kept);
            if (lane == 0) chunk_cnt[c] = tot;
        } else {
            const uint32_t kept = lane_cnt[c * kWave + lane];
            uint32_t pre = kept;  // kept edges of the lanes before this one
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const uint32_t u = __shfl_up(pre, o, kWave);
                if (lane >= o) pre += u;
            }
            uint64_t out = chunk_off[c] + (pre - kept);
            for (uint64_t m = starts; m; m &= m - 1) {
                uint32_t f = 0, to = 0;
                const int r = line(lo + (uint32_t)__builtin_ctzll(m), f, to);
                if (r > 0 && f != to) {
                    if (out < max_edges) {
                        src[out] = f;
                        dst[out] = to;
                        top = max(top, max(f, to));
                    }
                    out++;
                }
            }
        }
        parse_lds_sync();  // the next chunk overwrites the window
    }
    if (WRITE) {
        // most wavefronts find a larger id there already: atomics on one word
        // complete one after another (a pass over the pairs with one atomic per
        // wavefront took 190 us at 3M edges)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) top = max(top, (uint32_t)__shfl_xor((int)top, o, kWave));
        if (lane == 0 && top > ld_relaxed_agent(maxid)) atomicMax(maxid, top);
    }
}

template <typename C>
static void parse_layout(C &c, uint64_t nbytes, uint32_t **cnt, uint8_t **lanes, uint64_t **off, uint32_t **maxid,
                         unsigned long long **bad, void **sw, size_t *swb) {
    const uint64_t nchunks = (nbytes + kParseChunk - 1) / kParseChunk;
    *cnt = c.template take<uint32_t>(nchunks + 1);
    *lanes = c.template take<uint8_t>(nchunks * kWave + 1);
    *off = c.template take<uint64_t>(nchunks + 1);
    *maxid = c.template take<uint32_t>(1);
    *bad = c.template take<unsigned long long>(1);
    *swb = scan_workspace(nchunks + 1);
    *sw = c.template take<char>(*swb);
}

}  // namespace gchi

using namespace gchi;

extern "C" int gchi_parse_edgelist_workspace(uint64_t nbytes, size_t *bytes) {
    GCHI_CHECK(bytes, GCHI_ERR_INVALID, "null bytes");
    SizerAdapter a;
    uint32_t *cnt, *mx;
    uint8_t *lanes;
    uint64_t *off;
    unsigned long long *bad;
    void *sw;
    size_t swb;
    parse_layout(a, nbytes, &cnt, &lanes, &off, &mx, &bad, &sw, &swb);
    *bytes = a.z.off;
    return GCHI_OK;
}

extern "C" int gchi_parse_edgelist(const uint8_t *d_text, uint64_t nbytes, uint32_t *d_src, uint32_t *d_dst,
                                   uint64_t max_edges, uint64_t *h_nedges, uint32_t *h_maxid, void *d_work,
                                   size_t work_bytes, void *stream) {
    GCHI_CHECK(h_nedges && h_maxid && (nbytes == 0 || d_text), GCHI_ERR_INVALID, "parse_edgelist: null argument");
    GCHI_CHECK(max_edges == 0 || (d_src && d_dst), GCHI_ERR_INVALID, "parse_edgelist: null output");
    Carver c(d_work, work_bytes);
    uint32_t *cnt, *mx;
    uint8_t *lanes;
    uint64_t *off;
    unsigned long long *bad;
    void *sw;
    size_t swb;
    parse_layout(c, nbytes, &cnt, &lanes, &off, &mx, &bad, &sw, &swb);
    GCHI_CHECK(d_work && c.ok(), GCHI_ERR_WORKSPACE, "parse_edgelist: workspace too small");
    *h_nedges = 0;
    *h_maxid = 0;
    if (nbytes == 0) return GCHI_OK;
    hipStream_t s = as_stream(stream);
    const uint64_t nchunks = (nbytes + kParseChunk - 1) / kParseChunk;
    launch_fill_u32(mx, 0u, 1, s);
    launch_fill_u64(reinterpret_cast<uint64_t *>(bad), ~0ull, 1, s);
    const unsigned grid = grid_for(nchunks, kParseWaves, 1u << 15);
    hipLaunchKernelGGL(parse_pass<0>, dim3(grid), dim3(kParseWaves * kWave), 0, s, d_text, nbytes, nchunks,
                       cnt, lanes, off, d_src, d_dst, max_edges, bad, mx);
    GCHI_LAUNCH_CHECK();
    GCHI_TRY(exclusive_scan_u32_to_u64(cnt, off, nchunks, sw, swb, s));
    unsigned long long h_bad = 0;
    uint64_t total = 0;
    GCHI_HIP(hipMemcpyAsync(&h_bad, bad, 8, hipMemcpyDeviceToHost, s));
    GCHI_HIP(hipMemcpyAsync(&total, off + nchunks, 8, hipMemcpyDeviceToHost, s));
    GCHI_HIP(hipStreamSynchronize(s));
    if (h_bad != ~0ull)
        return fail(GCHI_ERR_FORMAT, "parse_edgelist: the line at byte " + std::to_string(h_bad) +
                                         " has fewer than two fields or is 1023 bytes or longer");
    *h_nedges = total;
    GCHI_CHECK(total <= max_edges || max_edges == 0, GCHI_ERR_INVALID, "parse_edgelist: more edges than max_edges");
    if (max_edges == 0 || total == 0) return GCHI_OK;
    hipLaunchKernelGGL(parse_pass<1>, dim3(grid), dim3(kParseWaves * kWave), 0, s, d_text, nbytes, nchunks,
                       cnt, lanes, off, d_src, d_dst, max_edges, bad, mx);
    GCHI_LAUNCH_CHECK();
    GCHI_HIP(hipMemcpyAsync(h_maxid, mx, 4, hipMemcpyDeviceToHost, s));
    GCHI_HIP(hipStreamSynchronize(s));
    return GCHI_OK;
}
