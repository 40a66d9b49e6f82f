// Entropy coder of the Falcons interpolation path on gfx950: the RleFseEncoder<int16_t> stream
// format (include/Falcons/encoder/RleFseEncoder.hpp) produced and consumed on the GPU.
//
//  method 0: runs of the zero code and the other codes as Elias-gamma classes (bytes) plus
//            MSB-first mantissa bits; the class bytes go through FSE in 64 K blocks.
//  method 1: order-1 tANS: per segment, 4 chunks, each one tANS chain whose table is switched per
//            symbol by the context of the previous code; codes with |code| >= 128 escape to a
//            gamma/FSE side stream.
//
// Data-parallel steps (sampling, delta, escape selection, context histograms, run/value extraction,
// mantissa bit packing, block framing, run expansion, prefix sums) run across the whole chip. The
// tANS and FSE chains are sequential state machines. They are cut into pieces, and what is followed
// through a piece is every state that may enter it, or a guess that is repaired; a walk picks the true
// ones. Chains that cannot be cut (decoding with many escapes) run in a workgroup each.
#include <cstdio>
#include <cstdlib>
#include <stdexcept>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <array>
#include <exception>
#include <thread>
#include <type_traits>

#include "fz_common.h"
#include "fz_fse.h"
#include "fz_kernels.h"
#include "fz_select.h"
#include "fz_split.h"

namespace fz {

constexpr int kO1K = 4;                  // RleFseEncoder.hpp:479
constexpr uint64_t kO1Seg = 8ull << 20;  // :577
constexpr uint32_t kFblk = 65536;        // :75

// Context bucket of the previous code (RleFseEncoder.hpp:354-385 in closed form): 0 for 0,
// magnitudes 1..4 one bucket each, then 5..7, 8..11 and >= 12; times two for the sign.
__host__ __device__ inline int o1_ctx(int code) {
    if (code == 0) return 0;
    const int sgn = code < 0;
    const int a = sgn ? -code : code;
    int m;
    if (a <= 4) m = a - 1;
    else if (a <= 7) m = 4;
    else if (a <= 11) m = 5;
    else m = 6;
    return 1 + 2 * m + sgn;
}
// Zigzag symbol clamped to 255 (escape).
__host__ __device__ inline int o1_sym(int code) {
    const uint32_t zz = ((uint32_t)code << 1) ^ (uint32_t)(code >> 31);
    return zz < 255 ? (int)zz : 255;
}

// LDS pointers carry their address space so that every access is an LDS instruction.
#define FZ_LDS __attribute__((address_space(3)))
template <typename T>
__device__ __forceinline__ FZ_LDS T* lds(T* p) { return (FZ_LDS T*)p; }
// Device-memory pointers likewise: global instructions count only in vmcnt, so loads issued ahead
// stay in flight across the LDS waits of a dependent chain (flat loads count in lgkmcnt as well).
#define FZ_GLB __attribute__((address_space(1)))
template <typename T>
__device__ __forceinline__ FZ_GLB T* glb(T* p) { return (FZ_GLB T*)p; }

// ---------------------------------------------------------------- small device helpers
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t uniform32(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
    return (uint64_t)uniform32((uint32_t)v) | (uint64_t)uniform32((uint32_t)(v >> 32)) << 32;
}

// LDS accesses of one wave on either side stay in order (the hardware keeps a wave's LDS operations in
// order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Backward reader with a 64-bit window in registers: bits [lo, lo + 64) of the stream (bytes below the
// start read as zero), refilled when a read reaches below lo; a refill covers at least 57 bits.
struct BitWin {
    const uint8_t* buf;
    int64_t pos;  // bits below pos are unread
    int64_t lo;
    uint64_t w;
};
__device__ __forceinline__ void bwin_fill(BitWin& r) {
    const int64_t b0 = (r.pos - 57) >> 3;  // floor for negatives
    // eight independent loads (addresses clamped, bytes below the start masked to zero) issued
    // together, so a refill costs one memory latency
    uint32_t v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = r.buf[b0 + j < 0 ? 0 : b0 + j];
    uint64_t w = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) w |= (uint64_t)(b0 + j < 0 ? 0u : v[j]) << (8 * j);
    r.w = w;
    r.lo = b0 * 8;
}
__device__ __forceinline__ BitWin bwin_at(const uint8_t* buf, int64_t pos) {
    BitWin r{buf, pos, 0, 0};
    bwin_fill(r);
    return r;
}
__device__ __forceinline__ uint32_t bwin_read(BitWin& r, uint32_t nb) {
    const int64_t p = r.pos - nb;
    if (p < r.lo) {
        r.pos = p + nb;
        bwin_fill(r);
    }
    r.pos = p;
    return nb ? (uint32_t)((r.w >> (p - r.lo)) & ((1ull << nb) - 1)) : 0u;
}

// ---------------------------------------------------------------- preprocess (RleFse:850-895)
struct PreCounts {
    unsigned long long z, zd, cnt, cntd;
};
__global__ void k_preprocess(const int16_t* bins, uint64_t n, uint64_t NW, uint64_t WL, uint64_t step, PreCounts* out) {
    __shared__ unsigned long long sz[256], szd[256], sc[256], scd[256];
    const uint64_t w = threadIdx.x;
    unsigned long long z = 0, zd = 0, c = 0, cd = 0;
    // windows are taken in order and the scan stops at the first one that does not fit
    if (w < NW) {
        bool fits = true;
        for (uint64_t v = 0; v <= w; v++)
            if (v * step + WL > n) { fits = false; break; }
        if (fits) {
            const uint64_t off = w * step;
            int16_t prev = bins[off];
            for (uint64_t t = 0; t < WL; t++) {
                const int16_t x = bins[off + t];
                z += (x == 0);
                if (t > 0 && x == prev) zd++;
                prev = x;
            }
            c = WL;
            cd = WL - 1;
        }
    }
    sz[threadIdx.x] = z; szd[threadIdx.x] = zd; sc[threadIdx.x] = c; scd[threadIdx.x] = cd;
    __syncthreads();
    if (threadIdx.x == 0) {
        PreCounts r{0, 0, 0, 0};
        for (int i = 0; i < 256; i++) { r.z += sz[i]; r.zd += szd[i]; r.cnt += sc[i]; r.cntd += scd[i]; }
        *out = r;
    }
}

__global__ void k_delta(const int16_t* __restrict__ in, int16_t* __restrict__ out, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = i ? (int16_t)(in[i] - in[i - 1]) : in[0];
}

static inline unsigned nblk(uint64_t n, unsigned bs = 256) { return (unsigned)((n + bs - 1) / bs); }

// ---------------------------------------------------------------- FSE tables (workgroup-wide)
// FSE symbol spread and table construction in LDS by a 256-thread workgroup, for any table log up
// to 13. Spread (zfse/fse_compress.c FSE_buildCTable_wksp, fse_decompress.c FSE_buildDTable):
// symbols with count -1 take the top positions in symbol order; the k-th occurrence of the others
// (in symbol order) goes to the k-th position of the walk j*step mod 2^tableLog, j = 0, 1, ...,
// that lies at or below the high threshold. The walk is a permutation (step is odd), so it is
// enumerated in parallel and ranked with a block scan. Within a symbol, positions in increasing
// order get consecutive states: each wave takes a quarter of the positions 64 at a time, and a
// position's place among its symbol's is the symbol's count in the quarters and steps before plus the
// lanes below that hold the same symbol (eight ballots). One thread per symbol scanning the whole
// table, and scans by one lane, took 0.54 ms for the 15 tables of one segment, as long for a small
// field as for a large one; this takes 0.04 ms.
template <unsigned MaxLog>
struct TableLdsT {
    int16_t norm[256];          // symbols above maxSym hold 0
    uint32_t cum[257];          // exclusive prefix of the counts (-1 counts as 1)
    uint32_t cump[257];         // exclusive prefix of the positive counts
    union {
        uint64_t part[4];       // scans: sums of the waves
        uint16_t wcnt[4][256];  // positions of each symbol in the quarters before, then so far
    };
    int32_t high;               // last position of the walk part; -1 when every count is -1
    int bad;
    uint8_t sym[1u << MaxLog];
};
using TableLds = TableLdsT<kFseMaxTableLog>;

// Exclusive prefix of v over the 256 threads of a workgroup; *total their sum. part: four words of LDS.
__device__ __forceinline__ uint64_t block_scan_u64(uint64_t v, uint64_t* part, uint64_t* total) {
    const unsigned t = threadIdx.x, l = t & 63u, w = t >> 6;
    uint64_t x = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint64_t o = __shfl_up((unsigned long long)x, d);
        if (l >= (unsigned)d) x += o;
    }
    __syncthreads();
    if (l == 63) part[w] = x;
    __syncthreads();
    uint64_t before = 0, sum = 0;
    for (unsigned i = 0; i < 4; i++) {
        if (i < w) before += part[i];
        sum += part[i];
    }
    __syncthreads();
    *total = sum;
    return before + x - v;
}

template <class TL>
__device__ bool spread_parallel(TL& L, unsigned tl) {
    const unsigned t = threadIdx.x;
    const uint32_t ts = 1u << tl, mask = ts - 1, step = (ts >> 1) + (ts >> 3) + 3;
    const int v = L.norm[t];
    // counts, positive counts and -1 counts in one scan (at most 256 * 2^13 each)
    const uint64_t cp = v > 0 ? (uint64_t)min(v, (int)ts) : 0u, low = v == -1 ? 1u : 0u;
    uint64_t sum;
    const uint64_t pre = block_scan_u64((cp + low) | cp << 22 | low << 44, L.part, &sum);
    constexpr uint64_t m22 = (1u << 22) - 1;
    L.cum[t] = (uint32_t)(pre & m22);
    L.cump[t] = (uint32_t)(pre >> 22 & m22);
    if (t == 0) {
        L.cum[256] = (uint32_t)(sum & m22);
        L.cump[256] = (uint32_t)(sum >> 22 & m22);
        L.high = (int32_t)ts - 1 - (int32_t)(sum >> 44);
    }
    if (__syncthreads_or(v < -1 || v > (int)ts || (sum & m22) != ts)) return false;
    if (low) L.sym[ts - 1 - (uint32_t)(pre >> 44)] = (uint8_t)t;
    const int32_t high = L.high;
    const uint32_t per = (ts + 255) / 256;  // walk steps per thread
    const uint32_t k0 = min(ts, t * per), k1 = min(ts, k0 + per);
    uint32_t rank = k0;
    if (high + 1 != (int32_t)ts) {
        uint32_t cnt = 0;
        for (uint32_t k = k0; k < k1; k++) cnt += (int32_t)((k * step) & mask) <= high;
        rank = (uint32_t)block_scan_u64(cnt, L.part, &sum);
    }
    int s = 0, hi = 256;  // last symbol with cump <= rank: the one whose counts hold rank
    while (hi - s > 1) {
        const int mid = (s + hi) >> 1;
        if (L.cump[mid] <= rank) s = mid; else hi = mid;
    }
    for (uint32_t k = k0; k < k1; k++) {
        const uint32_t pos = (k * step) & mask;
        if ((int32_t)pos > high) continue;
        while (s < 255 && L.cump[s + 1] <= rank) s++;
        L.sym[pos] = (uint8_t)s;
        rank++;
    }
    __syncthreads();
    return true;
}

// After spread_parallel: f(position, symbol, place of the position among its symbol's, in order).
template <class TL, class F>
__device__ __forceinline__ void rank_positions(TL& L, unsigned tl, F&& f) {
    const unsigned t = threadIdx.x, l = t & 63u, w = t >> 6;
    const uint32_t ts = 1u << tl, span = max(64u, ts / 4);
    const uint32_t u0 = min(ts, w * span), u1 = min(ts, u0 + span);
    // lanes of this step that hold the same symbol
    auto same = [&](uint32_t s, bool in) {
        uint64_t m = __ballot(in);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const uint64_t z = __ballot((s >> b) & 1u);
            m &= (s >> b) & 1u ? z : ~z;
        }
        return m;
    };
#pragma unroll
    for (int i = 0; i < 4; i++) L.wcnt[w][l + 64 * i] = 0;
    wave_lds_order();
    for (uint32_t u = u0; u < u1; u += 64) {
        const bool in = u + l < u1;
        const uint32_t s = in ? L.sym[u + l] : 0u;
        const uint64_t m = same(s, in);
        if (in && (m & ((1ull << l) - 1)) == 0) L.wcnt[w][s] = (uint16_t)(L.wcnt[w][s] + __popcll(m));
        wave_lds_order();
    }
    __syncthreads();
    {
        uint32_t acc = 0;
        for (int i = 0; i < 4; i++) {
            const uint32_t n = L.wcnt[i][t];
            L.wcnt[i][t] = (uint16_t)acc;
            acc += n;
        }
    }
    __syncthreads();
    for (uint32_t u = u0; u < u1; u += 64) {
        const bool in = u + l < u1;
        const uint32_t s = in ? L.sym[u + l] : 0u;
        const uint64_t m = same(s, in);
        const uint64_t before = m & ((1ull << l) - 1);
        const uint32_t base = L.wcnt[w][s];
        wave_lds_order();
        if (in && before == 0) L.wcnt[w][s] = (uint16_t)(base + __popcll(m));
        wave_lds_order();
        if (in) f(u + l, s, base + (uint32_t)__popcll(before));
    }
}

// FSE_buildCTable_wksp (fse_compress.c:65-155) after spread_parallel; thread t handles symbol t.
template <class TL, class CT>
__device__ void ctable_parallel(TL& L, unsigned tl, unsigned maxSym, CT* ct) {
    const unsigned t = threadIdx.x;
    const uint32_t ts = 1u << tl;
    const int nc = L.norm[t];
    rank_positions(L, tl, [&](uint32_t u, uint32_t s, uint32_t r) { ct->stateTable[L.cum[s] + r] = (uint16_t)(ts + u); });
    if (nc == 0) {
        ct->deltaNbBits[t] = ((tl + 1) << 16) - ts;
        ct->deltaFindState[t] = 0;
    } else if (nc == -1 || nc == 1) {
        ct->deltaNbBits[t] = (tl << 16) - ts;
        ct->deltaFindState[t] = (int32_t)L.cum[t] - 1;
    } else {
        const uint32_t maxBitsOut = tl - highbit32((uint32_t)(nc - 1));
        ct->deltaNbBits[t] = (maxBitsOut << 16) - ((uint32_t)nc << maxBitsOut);
        ct->deltaFindState[t] = (int32_t)L.cum[t] - nc;
    }
    if (t == 0) { ct->tableLog = tl; ct->maxSym = maxSym; }
}

// FSE_buildDTable (fse_decompress.c:70-127) after spread_parallel. entry(symbol) goes into the top
// four bits of nbBits.
template <class TL, class X>
__device__ void dtable_parallel(TL& L, unsigned tl, DEntry* dt, X&& extra) {
    const uint32_t ts = 1u << tl;
    rank_positions(L, tl, [&](uint32_t u, uint32_t s, uint32_t r) {
        const int nc = L.norm[s];
        const uint32_t ns = (nc == -1 ? 1u : (uint32_t)nc) + r;
        const uint32_t nb = tl - highbit32(ns);
        dt[u] = DEntry{(uint16_t)((ns << nb) - ts), (uint8_t)s, (uint8_t)(nb | extra(s) << 4)};
    });
}
template <class TL>
__device__ void dtable_parallel(TL& L, unsigned tl, DEntry* dt) {
    dtable_parallel(L, tl, dt, [](uint32_t) { return 0u; });
}

// ---------------------------------------------------------------- FSE block (workgroup-wide)
// FSE_compress of blocks of at most 64 K bytes (fse_compress.c:632-694), framed as in RleFse:150-176:
// [0][raw] | [2][sym] | [1][u32 len][FSE bytes].
// FSE_compress bounds the table log by FSE_DEFAULT_TABLELOG (11).
//
// The encode (fse_compress.c:578-628) emits symbols n-3 down to 0 alternately from two states, the
// first of them seeded by symbol n-1 and the second by n-2 (in zfse's names: state 2 then state 1
// for an even n, state 1 then state 2 for an odd one), then state 2's and state 1's final values
// (tl bits each) and the end mark; the bytes are those bits LSB-first. A lane that follows each state
// through its half of the symbols needs 32,768 dependent table steps of 80 ns for a block of 64 K.
// Runs from two states under the same symbols do not soon become one (after 1,500 steps for the
// classes of escaped codes, 12,000 for five equally frequent symbols), but after a symbol of count c
// only c states of 2,048 are left, and a few dozen 300 steps on. So the two chains are cut into pieces of
// 1,024 steps, a wave follows all states that a symbol in front of its piece leaves, one a lane at the
// piece (k_fse_sets), and a walk from piece to piece picks the true ones, with the bits of every 128
// steps noted on the way (k_fse_finish, which then writes the bits, 256 lanes a block). A piece that
// more than 64 states reach (two symbols of equal counts: no two states ever meet) is run by the walk.
// Escape classes of a 512^3 k^-3 field (one workgroup a block, two lanes at work -> these kernels): REL 1e-3, 14 blocks
// (50,000 escapes), 2.06 -> 0.37 ms; 3.3e-4, 99 blocks (6 million), 2.75 -> 1.98, of which the walk 1.16: some
// blocks hardly have a set; 1e-4, 1,036 blocks (67 million), 4.42 -> 2.1, the waves' LDS reads by then. One block of
// 35,000: 1.29 -> 0.23. Pieces of 512 steps run half as many steps twice: 765 full blocks 2.4 ms against 1.9.
constexpr unsigned kFblkLog = kFseDefaultTableLog;
constexpr uint32_t kFseGroup = 16;      // symbols of a load
constexpr uint32_t kFseHists = 8;
constexpr uint32_t kFseSub = 128;       // steps of a chain between noted states
constexpr uint32_t kFsePiece = 1024;    // steps of a chain in a piece
constexpr uint32_t kFseSubs = kFblk / (2 * kFseSub), kFsePieces = kFblk / (2 * kFsePiece);
constexpr uint32_t kFseFields = kFsePiece / kFseSub + 1;
constexpr uint32_t kFseWarm = 448;      // steps in front of a piece; the first 128 are searched
constexpr uint32_t kFseSearch = 128;
constexpr uint32_t kFseWarmFew = 704;   // up to here for a symbol of a count up to 256, then up to 1,024
constexpr uint32_t kFseWarmMax = 8192;  // how far back the search goes
constexpr uint32_t kFseLogWords = 2 * kFsePieces * kFseFields * 64;  // a block's noted states
constexpr uint64_t kFsePending = ~1ull;

// One FSE block of a batch: its input (class bytes, or a framed block to decode), its output and
// its length in symbols (at most 64 K).
struct FseBlk {
    const uint8_t* src;
    uint8_t* dst;
    uint32_t len, pad;
};

// What the kernels of a block hand on. result: 0 (not compressible), 1 (one symbol), kFseErr, or kFsePending.
struct FseMeta {
    CTableT<kFblkLog> ct;
    uint64_t result;
    uint32_t nc, tl;  // header bytes, table log
};

// 16 symbols ending below symbol h, the last of them in byte 15 (below symbol 0: zeros, not used).
__device__ __forceinline__ void fse_group(const uint8_t* src, uint32_t h, uint32_t (&w)[4]) {
    if (h >= kFseGroup) {
        __builtin_memcpy(w, src + h - kFseGroup, kFseGroup);
    } else {
        w[0] = w[1] = w[2] = w[3] = 0;
        for (uint32_t j = 0; j < h; j++) {
            const uint32_t at = kFseGroup - h + j, v = (uint32_t)src[j] << (8 * (at & 3u));
            w[0] |= at < 4 ? v : 0u;
            w[1] |= at >= 4 && at < 8 ? v : 0u;
            w[2] |= at >= 8 && at < 12 ? v : 0u;
            w[3] |= at >= 12 ? v : 0u;
        }
    }
}

// Both chains over the symbols hi - 1 down to lo (hi - lo a multiple of 16, or lo == 0), the first
// of them on chain 0. sink(value, bits) takes every emission in its order.
template <class F>
__device__ __forceinline__ void fse_run(const uint8_t* src, uint32_t hi, uint32_t lo, const CTableT<kFblkLog>& ct,
                                        uint32_t& s0, uint32_t& s1, F&& sink) {
    const FZ_LDS uint32_t* dnb = lds(ct.deltaNbBits);
    const FZ_LDS int32_t* dfs = lds(ct.deltaFindState);
    const FZ_LDS uint16_t* stt = lds(ct.stateTable);
    uint32_t cur[4], nxt[4];
    fse_group(src, hi, nxt);
    for (uint32_t h = hi; h > lo;) {
        const uint32_t cnt = min(h - lo, kFseGroup);
#pragma unroll
        for (int r = 0; r < 4; r++) cur[r] = nxt[r];
        h -= cnt;
        if (h > lo) fse_group(src, h, nxt);
        auto pair = [&](uint32_t a, uint32_t b, bool two) {
            const uint32_t n0 = (s0 + dnb[a]) >> 16;
            sink(s0, n0);
            s0 = stt[(s0 >> n0) + dfs[a]];
            if (two) {
                const uint32_t n1 = (s1 + dnb[b]) >> 16;
                sink(s1, n1);
                s1 = stt[(s1 >> n1) + dfs[b]];
            }
        };
        if (cnt == kFseGroup) {
#pragma unroll
            for (int r = 3; r >= 0; r--) {
                pair(cur[r] >> 24, cur[r] >> 16 & 255u, true);
                pair(cur[r] >> 8 & 255u, cur[r] & 255u, true);
            }
        } else {  // the block's last symbols
            for (uint32_t k = 0; k < cnt; k += 2) {
                const uint32_t at = kFseGroup - 1 - k;  // odd: both bytes in one word
                const uint32_t r = at >> 2, w = r == 3 ? cur[3] : r == 2 ? cur[2] : r == 1 ? cur[1] : cur[0];
                pair(w >> (8 * (at & 3u)) & 255u, w >> (8 * (at & 3u) - 8) & 255u, k + 1 < cnt);
            }
        }
    }
}

// Histogram, normalization, table header (to the block's slot) and encoding table of a block, by a
// workgroup; normalization and header by lane 0 (a class stream has few symbols).
__global__ void __launch_bounds__(256) k_fse_tables(const FseBlk* blks, uint8_t* slots, uint64_t slot, FseMeta* meta) {
    __shared__ union {
        uint32_t hist[kFseHists][256];  // one for every eighth lane: fewer adds to one word
        TableLdsT<kFblkLog> tab;
    } L;
    __shared__ uint32_t count[256];
    __shared__ CTableT<kFblkLog> ct;
    __shared__ uint64_t result;
    __shared__ uint32_t max_sym, log, head;
    const uint8_t* src = blks[blockIdx.x].src;
    const uint32_t n = blks[blockIdx.x].len, t = threadIdx.x;
    FseMeta& M = meta[blockIdx.x];
    for (uint32_t i = t; i < kFseHists * 256; i += blockDim.x) L.hist[i >> 8][i & 255u] = 0;
    __syncthreads();
    for (uint32_t i = t * kFseGroup; i < n; i += blockDim.x * kFseGroup) {
        uint32_t* hist = L.hist[t & (kFseHists - 1)];
        if (i + kFseGroup <= n) {
            uint32_t w[4];
            __builtin_memcpy(w, src + i, kFseGroup);
#pragma unroll
            for (int r = 0; r < 16; r++) atomicAdd(&hist[w[r >> 2] >> (8 * (r & 3)) & 255u], 1u);
        } else {
            for (uint32_t j = i; j < n; j++) atomicAdd(&hist[src[j]], 1u);
        }
    }
    __syncthreads();
    uint32_t c = 0;
    for (uint32_t k = 0; k < kFseHists; k++) c += L.hist[k][t];
    count[t] = c;
    __syncthreads();
    if (t == 0) {
        uint64_t r = kFsePending;
        head = log = max_sym = 0;
        if (n <= 1) {
            r = 0;
        } else {
            unsigned maxSym = 255;
            while (!count[maxSym]) maxSym--;
            uint32_t maxCount = 0;
            for (unsigned s = 0; s <= maxSym; s++) maxCount = count[s] > maxCount ? count[s] : maxCount;
            if (maxCount == n) r = 1;
            else if (maxCount == 1 || maxCount < (n >> 7)) r = 0;
            else {
                const unsigned tl = optimal_table_log(kFseDefaultTableLog, n, maxSym);
                for (unsigned s = maxSym + 1; s < 256; s++) L.tab.norm[s] = 0;
                if (tl > kFblkLog || normalize_count(L.tab.norm, tl, count, n, maxSym) == kFseErr) {
                    r = kFseErr;
                } else {
                    head = (uint32_t)write_ncount(slots + blockIdx.x * slot + 5, L.tab.norm, maxSym, tl);
                    log = tl;
                    max_sym = maxSym;
                }
            }
        }
        result = r;
    }
    __syncthreads();
    if (result == kFsePending) {
        if (spread_parallel(L.tab, log)) {
            ctable_parallel(L.tab, log, max_sym, &ct);
            __syncthreads();
            const uint32_t* from = reinterpret_cast<const uint32_t*>(&ct);
            uint32_t* to = reinterpret_cast<uint32_t*>(&M.ct);
            for (uint32_t i = t; i < sizeof(ct) / 4; i += blockDim.x) to[i] = from[i];
        } else {  // cannot happen for counts from normalize_count
            __syncthreads();
            if (t == 0) result = kFseErr;
            __syncthreads();
        }
    }
    if (t == 0) {
        M.result = result;
        M.nc = head;
        M.tl = log;
    }
}

__device__ __forceinline__ void fse_stage_table(CTableT<kFblkLog>& ct, const FseMeta& M) {
    const uint32_t* from = reinterpret_cast<const uint32_t*>(&M.ct);
    uint32_t* to = reinterpret_cast<uint32_t*>(&ct);
    for (uint32_t i = threadIdx.x; i < sizeof(ct) / 4; i += blockDim.x) to[i] = from[i];
    __syncthreads();
}

// Steps t0 up to t1 of a chain (step t codes symbol top[-2t]) for the R states of every lane: the lanes
// look up 64 steps at once (their symbols do not depend on the states), the next 64 symbols in flight.
template <int R>
__device__ __forceinline__ void fse_set_run(const uint8_t* top, uint32_t t0, uint32_t t1, const CTableT<kFblkLog>& ct,
                                            uint32_t (&st)[R], uint32_t& bits) {
    if (t0 >= t1) return;
    const uint32_t lane = threadIdx.x & 63u;
    const FZ_LDS uint32_t* dnb = lds(ct.deltaNbBits);
    const FZ_LDS int32_t* dfs = lds(ct.deltaFindState);
    const FZ_LDS uint16_t* stt = lds(ct.stateTable);
    auto load = [&](uint32_t t) { return (uint32_t)glb(top)[-2 * (int64_t)min(t + lane, t1 - 1)]; };
    uint32_t next = load(t0);
    for (uint32_t t = t0; t < t1; t += 64) {
        const uint32_t d = dnb[next];
        const int32_t f = dfs[next];
        if (t + 64 < t1) next = load(t + 64);
        auto step = [&](int k) {
            const uint32_t dk = (uint32_t)__builtin_amdgcn_readlane((int)d, k);
            const int32_t fk = __builtin_amdgcn_readlane(f, k);
#pragma unroll
            for (int r = 0; r < R; r++) {
                const uint32_t nb = (st[r] + dk) >> 16;
                if (r == 0) bits += nb;
                st[r] = stt[(int32_t)(st[r] >> nb) + fk];
            }
        };
        const int cnt = (int)min(t1 - t, 64u);
        if (cnt == 64 && R == 1) {
#pragma unroll 16
            for (int k = 0; k < 64; k++) step(k);
        } else {
            for (int k = 0; k < cnt; k++) step(k);
        }
    }
}

// The different ones of a wave's states (at least 1 << tl, below twice that), Q a lane, the last one filling
// the lanes left over. map: 64 words, list: 64 * Q states of LDS. False when there are more than that.
template <int R, int Q>
__device__ __forceinline__ bool fse_set_merge(const uint32_t (&st)[R], uint32_t (&out)[Q], uint32_t tl, FZ_LDS uint32_t* map,
                                              FZ_LDS uint16_t* list) {
    const uint32_t lane = threadIdx.x & 63u;
    map[lane] = 0;
    wave_lds_order();
#pragma unroll
    for (int r = 0; r < R; r++) {
        const uint32_t x = st[r] - (1u << tl);
        __hip_atomic_fetch_or(&map[x >> 5], 1u << (x & 31u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    wave_lds_order();
    uint32_t w = map[lane], inc = __popc(w);
    const uint32_t own = inc;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(inc, d, 64);
        if (lane >= d) inc += y;
    }
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)inc, 63);
    if (total > 64 * Q) return false;
    for (uint32_t at = inc - own; w; w &= w - 1) list[at++] = (uint16_t)((1u << tl) + lane * 32 + __ffs(w) - 1);
    wave_lds_order();
#pragma unroll
    for (int r = 0; r < Q; r++) out[r] = list[min(r * 64 + lane, total - 1)];
    wave_lds_order();
    return true;
}

// The steps t0 up to t1 of a piece: every lane's state at the start, after each 128 steps and at the end, with
// the bits of those steps.
__device__ __forceinline__ void fse_log_piece(const uint8_t* top, uint32_t t0, uint32_t t1, const CTableT<kFblkLog>& ct,
                                              uint32_t (&st)[1], uint32_t* log) {
    for (uint32_t f = 0; f + 1 < kFseFields && t0 + f * kFseSub < t1; f++) {
        const uint32_t at = st[0];
        uint32_t bits = 0;
        fse_set_run(top, t0 + f * kFseSub, min(t1, t0 + (f + 1) * kFseSub), ct, st, bits);
        log[f * 64] = at | bits << 16;
    }
    log[(kFseFields - 1) * 64] = st[0];
}

// A wave a piece of a chain (grid: blocks, pieces of both chains / 4). Bound by the latency of the steps' LDS reads.
__global__ void __launch_bounds__(256) k_fse_sets(const FseBlk* blks, const FseMeta* meta, uint32_t* logs) {
    __shared__ CTableT<kFblkLog> ct;
    __shared__ uint32_t maps[4][64];
    __shared__ uint16_t lists[4][256];
    const uint32_t b = blockIdx.x, lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const uint32_t unit = uniform32(blockIdx.y * 4u + wv), k = unit & 1u, p = unit >> 1;
    const uint32_t n = blks[b].len;
    // n >= 3 where a result is pending; a chain's steps are the emissions k, k + 2, ... below n - 2
    if (meta[b].result != kFsePending || blockIdx.y * 2u * kFsePiece >= (n - 1) / 2) return;
    const uint32_t tl = meta[b].tl;
    fse_stage_table(ct, meta[b]);
    const uint32_t steps = (n - 1 - k) / 2, t0 = p * kFsePiece, t1 = min(steps, t0 + kFsePiece);
    if (t0 >= steps) return;
    const uint8_t* src = blks[b].src;
    const uint8_t* top = src + (n - 3 - k);
    FZ_LDS uint32_t* map = lds(maps[wv]);
    FZ_LDS uint16_t* list = lds(lists[wv]);
    uint32_t* log = logs + (uint64_t)b * kFseLogWords + (k * kFsePieces + p) * kFseFields * 64 + lane;
    uint32_t st[1], from = 0, bits = 0;  // from: the first step that is left to run with one state a lane
    bool found = false;
    for (uint32_t warm = kFseWarm; !found;) {
        if (t0 <= warm) {  // from the block's end, where the state is known
            st[0] = init_state2(&ct, src[n - 1 - k]);
            from = 0;
            break;
        }
        if (warm > kFseWarmMax) {
            log[0] = 0;  // no state is 0: the walk runs this piece
            return;
        }
        uint32_t best = ~0u;
#pragma unroll
        for (uint32_t h = 0; h < kFseSearch; h += 64) {
            const uint32_t d = ct.deltaNbBits[top[-2 * (int64_t)(t0 - warm + h + lane)]];
            const uint32_t mb = (d >> 16) + 1;  // d = (mb << 16) - (c << mb)
            best = min(best, ((mb << 16) - d) >> mb << 8 | (h + lane));
        }
#pragma unroll
        for (uint32_t d = 32; d; d >>= 1) best = min(best, (uint32_t)__shfl_xor((int)best, (int)d, 64));
        best = uniform32(best);
        const uint32_t c = best >> 8;
        if (c > (warm <= kFseWarmFew ? 256u : 1024u)) {
            warm += kFseSearch;
            continue;
        }
        // the c states that the symbol of step from - 1 leaves
        from = t0 - warm + (best & 255u) + 1;
        const uint16_t* image = ct.stateTable + (ct.deltaFindState[top[-2 * (int64_t)(from - 1)]] + (int32_t)c);
        if (c <= 64) {
            st[0] = image[min(lane, c - 1)];
            break;
        }
        uint32_t s4[4];
        bool room = true;
        if (c <= 256) {
#pragma unroll
            for (uint32_t r = 0; r < 4; r++) s4[r] = image[min(r * 64 + lane, c - 1)];
        } else {
            uint32_t s16[16];
#pragma unroll
            for (uint32_t r = 0; r < 16; r++) s16[r] = image[min(r * 64 + lane, c - 1)];
            fse_set_run(top, from, from + 64, ct, s16, bits);  // at least 320 steps in front of the piece
            from += 64;
            room = fse_set_merge(s16, s4, tl, map, list);
        }
        while (room && !found && from < t0) {
            const uint32_t to = min(from + 256, t0);
            fse_set_run(top, from, to, ct, s4, bits);
            from = to;
            found = fse_set_merge(s4, st, tl, map, list);
        }
        warm *= 2;  // more than 64 are left: from further back
    }
    fse_set_run(top, from, t0, ct, st, bits);
    fse_log_piece(top, t0, t1, ct, st, log);
}
static_assert(kFseWarm >= kFseSearch + 64 + 256, "the merging runs end in front of the piece");

// A workgroup a block: the true states of both chains at every 256 symbols, the bits' places, the bits,
// the frame. sizes: the framed length.
__global__ void __launch_bounds__(256) k_fse_finish(const FseBlk* blks, const FseMeta* meta, uint32_t* logs,
                                                    uint8_t* slots, uint64_t slot, uint64_t* sizes) {
    __shared__ CTableT<kFblkLog> ct;
    __shared__ uint64_t scan[4];
    __shared__ uint32_t sub_state[kFseSubs], sub_bits[kFseSubs];  // states: chain 0 low, chain 1 high
    __shared__ uint32_t fin[2];
    __shared__ uint8_t pick[2][kFsePieces];
    const uint32_t b = blockIdx.x, t = threadIdx.x, lane = t & 63u, wv = t >> 6;
    const uint8_t* src = blks[b].src;
    const uint32_t n = blks[b].len;
    uint8_t* out = slots + b * slot;
    uint8_t* fo = out + 5;
    uint64_t r = meta[b].result;
    const uint32_t tl = meta[b].tl, nc = meta[b].nc;
    if (r == kFsePending) {
        fse_stage_table(ct, meta[b]);
        const uint32_t m = n - 2;  // emissions: symbols n - 3 .. 0
        if (wv < 2) {
            const uint32_t k = wv, steps = (m - k + 1) / 2, np = (steps + kFsePiece - 1) / kFsePiece;
            uint32_t* log = logs + (uint64_t)b * kFseLogWords + k * kFsePieces * kFseFields * 64 + lane;
            uint32_t cur = uniform32(init_state2(&ct, src[n - 1 - k]));
            for (uint32_t p0 = 0; p0 < np; p0 += 8) {
                uint32_t s[8], e[8];
#pragma unroll
                for (uint32_t j = 0; j < 8; j++) {
                    const uint32_t p = min(p0 + j, np - 1);
                    s[j] = log[p * kFseFields * 64];
                    e[j] = log[(p * kFseFields + kFseFields - 1) * 64];
                }
#pragma unroll
                for (uint32_t j = 0; j < 8; j++) {
                    if (p0 + j < np) {
                        const uint64_t hit = __ballot((s[j] & 0xFFFFu) == cur);
                        const uint32_t w = hit ? (uint32_t)__ffsll((unsigned long long)hit) - 1u : 0u;
                        if (lane == 0) pick[k][p0 + j] = (uint8_t)w;
                        if (hit) {
                            cur = (uint32_t)__builtin_amdgcn_readlane((int)e[j], (int)w) & 0xFFFFu;
                        } else {  // a piece without a set
                            uint32_t st[1] = {cur};
                            const uint32_t t0 = (p0 + j) * kFsePiece;
                            fse_log_piece(src + (n - 3 - k), t0, min(steps, t0 + kFsePiece), ct, st,
                                          log + (p0 + j) * kFseFields * 64);
                            cur = uniform32(st[0]);
                        }
                    }
                }
            }
            if (lane == 0) fin[k] = cur;
        }
        __syncthreads();
        const uint32_t hi = t * 2 * kFseSub < m ? m - t * 2 * kFseSub : 0u, lo = hi > 2 * kFseSub ? hi - 2 * kFseSub : 0u;
        if (hi) {
            uint32_t w[2] = {0, 0};
            for (uint32_t k = 0; k < 2; k++) {
                const uint32_t p = t / (kFseFields - 1), f = t % (kFseFields - 1);
                if (t * kFseSub < (m - k + 1) / 2)  // m odd: chain 1 can end a piece earlier
                    w[k] = logs[(uint64_t)b * kFseLogWords + ((k * kFsePieces + p) * kFseFields + f) * 64 + pick[k][p]];
            }
            sub_state[t] = (w[0] & 0xFFFFu) | w[1] << 16;
            sub_bits[t] = (w[0] >> 16) + (w[1] >> 16);
        }
        __syncthreads();
        uint64_t sbits;
        const uint64_t off0 = block_scan_u64(hi ? sub_bits[t] : 0u, scan, &sbits);
        const uint64_t total = nc + (sbits + 2 * (uint64_t)tl + 1 + 7) / 8;
        r = total >= n - 1 ? 0 : total;
        if (r) {
            // Bits go to whole words from the last word boundary at or before the stream (the header's
            // last bytes share it). A lane stores the words that only it reaches; a word that two lanes
            // share is cleared first and takes its parts by atomics, as do those of the closing states.
            uint8_t* sb = fo + nc;
            const uint32_t lead = (uint32_t)((uintptr_t)sb & 3u);
            uint32_t* wbase = reinterpret_cast<uint32_t*>(sb - lead);
            const uint64_t off = off0 + 8 * lead, fin_bit = sbits + 8 * lead;
            uint32_t head = 0;
            if (t == 0)
                for (uint32_t k = 0; k < lead && k < nc; k++) head |= (uint32_t)fo[nc - 1 - k] << (8 * (lead - 1 - k));
            __syncthreads();
            if (hi) wbase[off >> 5] = 0;
            if (t == 0) {
                const uint64_t last = (fin_bit + 2 * tl) >> 5;
                for (uint64_t w = fin_bit >> 5; w <= last; w++) wbase[w] = 0;
            }
            __syncthreads();
            if (t == 0 && lead) atomicOr(&wbase[0], head);
            if (hi) {
                uint32_t s0 = sub_state[t] & 0xFFFFu, s1 = sub_state[t] >> 16;
                uint64_t acc = 0;
                uint32_t have = (uint32_t)(off & 31u);
                uint32_t* wp = wbase + (off >> 5);
                bool first = true;  // the word is shared with the lane before
                fse_run(src, hi, lo, ct, s0, s1, [&](uint32_t v, uint32_t nb) {
                    acc |= (uint64_t)(v & ((1u << nb) - 1u)) << have;
                    have += nb;
                    if (have >= 32) {
                        if (first) atomicOr(wp, (uint32_t)acc);
                        else *wp = (uint32_t)acc;
                        first = false;
                        wp++;
                        acc >>= 32;
                        have -= 32;
                    }
                });
                if (have && (uint32_t)acc) atomicOr(wp, (uint32_t)acc);  // shared with the lane after
            }
            if (t == 0) {
                const uint32_t f0 = fin[n & 1u], f1 = fin[(n & 1u) ^ 1u];  // state 2 is chain 0 for an even n
                const uint32_t mask = (1u << tl) - 1u, sh = (uint32_t)(fin_bit & 31u);
                const uint64_t v = (uint64_t)(f0 & mask) | (uint64_t)(f1 & mask) << tl | 1ull << (2 * tl);
                atomicOr(&wbase[fin_bit >> 5], (uint32_t)(v << sh));
                if (sh + 2 * tl + 1 > 32) atomicOr(&wbase[(fin_bit >> 5) + 1], (uint32_t)(v << sh >> 32));
            }
        }
    }
    if (r == kFseErr || r == 0 || r >= n) {
        if (t == 0) {
            out[0] = 0;
            sizes[b] = 1 + n;
        }
        for (uint32_t i = t; i < n; i += blockDim.x) out[1 + i] = src[i];
    } else if (r == 1) {
        if (t == 0) {
            out[0] = 2;
            out[1] = src[0];
            sizes[b] = 2;
        }
    } else if (t == 0) {
        out[0] = 1;
        for (uint32_t k = 0; k < 4; k++) out[1 + k] = (uint8_t)((uint32_t)r >> (8 * k));
        sizes[b] = 5 + r;
    }
}

// Copies variable-size slots to their packed places (blks[b].dst, found by the host from the sizes).
__global__ void k_pack_slots(const uint8_t* slots, uint64_t slot_stride, const uint64_t* sizes, const FseBlk* blks) {
    const uint64_t b = blockIdx.y;
    const uint64_t sz = sizes[b];
    uint8_t* out = blks[b].dst;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < sz; i += (uint64_t)gridDim.x * blockDim.x)
        out[i] = slots[b * slot_stride + i];
}

// FSE_decompress of one block (fse_decompress.c:254-282): the workgroup reads the header and builds
// the decoding table; lane 0 decodes. Tables up to log 11 (all that FSE_compress writes) run with
// the compressed bytes and the decoded bytes in LDS, copied in and out by the whole workgroup;
// logs 12 and 13 read and write device memory directly.
struct FseDecSmall {  // about 75 KB: two workgroups to a CU
    TableLdsT<kFblkLog> tab;
    DEntry dt[1u << kFblkLog];
    alignas(16) uint8_t in[kFblk + 64];
};
struct FseDecBig {
    TableLdsT<kFseMaxTableLog> tab;
    DEntry dt[1u << kFseMaxTableLog];
};
struct FseDecLds {
    union {
        FseDecSmall s;
        FseDecBig g;
    };
    int16_t norm[256];
    uint32_t tl;
    uint64_t hl;
};

// The two-state FSE decode loop (fse_decompress.c:254-282 via FSE_decompress_usingDTable).
// The two states decode alternate symbols; their table entries are read together.
__device__ __forceinline__ void fse_decode_run(const DEntry* dt, const uint8_t* bs, uint64_t bsz, unsigned tl,
                                               uint8_t* dst, uint32_t len) {
    BitWin r = bwin_at(bs, (int64_t)(bsz - 1) * 8 + (int64_t)highbit32(bs[bsz - 1]));
    uint32_t s0 = bwin_read(r, tl);
    uint32_t s1 = bwin_read(r, tl);
    uint32_t i = 0;
    for (; i + 2 <= len; i += 2) {
        const DEntry e0 = dt[s0], e1 = dt[s1];
        dst[i] = e0.symbol;
        dst[i + 1] = e1.symbol;
        s0 = e0.newState + bwin_read(r, e0.nbBits);
        s1 = e1.newState + bwin_read(r, e1.nbBits);
    }
    if (i < len) dst[i] = dt[s0].symbol;
}

// The same loop with the table and the bitstream in LDS (in: the bitstream, bsz bytes, 4-byte
// aligned with 12 readable bytes past its end); the symbols go to out in device memory (4-byte
// aligned), four to a store. The bits below the read position sit in a 64-bit buffer refilled from
// aligned LDS words once per two symbol pairs (two pairs read at most 4 * 11 bits); the state values
// stay in vector registers.
__device__ __forceinline__ void fse_decode_run_lds(const FZ_LDS DEntry* dt, const FZ_LDS uint8_t* in, uint64_t bsz,
                                                   unsigned tl, uint8_t* out, uint32_t len) {
    const FZ_LDS uint32_t* w32 = reinterpret_cast<const FZ_LDS uint32_t*>(in);
    // entries as words: [15:0] next state base, [23:16] symbol, [31:24] bit count
    const FZ_LDS uint32_t* dtw = reinterpret_cast<const FZ_LDS uint32_t*>(dt);
    int32_t p = (int32_t)((bsz - 1) * 8) + (int32_t)highbit32(in[bsz - 1]);
    uint64_t buf = 0;
    int32_t prel = 0;
    auto refill = [&]() {  // bits [p - prel, p); bytes below the start read as zero
        const int32_t lo = p - 64;
        const int32_t lc = max(lo, 0);
        const int32_t j0 = lc >> 5;
        const uint32_t sh = (uint32_t)lc & 31u;
        uint64_t b = (uint64_t)__builtin_amdgcn_alignbit(w32[j0 + 1], w32[j0], sh) |
                     ((uint64_t)__builtin_amdgcn_alignbit(w32[j0 + 2], w32[j0 + 1], sh) << 32);
        if (lo < 0) b = (p > 0 ? b << (uint32_t)(-lo) : 0ull);  // move bit p-1 to the top, zeros below
        buf = b;
        prel = 64;
        (void)lo;
    };
    auto read = [&](uint32_t nb) -> uint32_t {
        prel -= (int32_t)nb;
        p -= (int32_t)nb;
        return (uint32_t)(buf >> ((uint32_t)prel & 63u)) & ((1u << nb) - 1u);
    };
    refill();
    uint32_t s0 = read(tl);
    uint32_t s1 = read(tl);
    uint32_t i = 0;
    for (; i + 4 <= len; i += 4) {
        refill();
        const uint32_t e0 = dtw[s0], e1 = dtw[s1];
        s0 = (e0 & 0xFFFFu) + read(e0 >> 24);
        s1 = (e1 & 0xFFFFu) + read(e1 >> 24);
        const uint32_t f0 = dtw[s0], f1 = dtw[s1];
        s0 = (f0 & 0xFFFFu) + read(f0 >> 24);
        s1 = (f1 & 0xFFFFu) + read(f1 >> 24);
        const uint32_t v = ((e0 >> 16) & 0xFFu) | (((e1 >> 16) & 0xFFu) << 8) | (((f0 >> 16) & 0xFFu) << 16) |
                           (((f1 >> 16) & 0xFFu) << 24);
        *reinterpret_cast<uint32_t*>(out + i) = v;
    }
    for (; i + 2 <= len; i += 2) {
        refill();
        const uint32_t e0 = dtw[s0], e1 = dtw[s1];
        out[i] = (uint8_t)(e0 >> 16);
        out[i + 1] = (uint8_t)(e1 >> 16);
        s0 = (e0 & 0xFFFFu) + read(e0 >> 24);
        s1 = (e1 & 0xFFFFu) + read(e1 >> 24);
    }
    if (i < len) out[i] = (uint8_t)(dtw[s0] >> 16);
}

// The layout for launches whose blocks all have tables up to log 11 (all that FSE_compress writes):
// the bitstream is staged kFseWin bytes at a time, so that a workgroup takes about 31 KB of LDS and
// five run on a CU (a launch of 1,036 blocks, the escape streams of a 512^3 REL 1e-4 field, then
// runs in one wave of workgroups instead of three).
constexpr uint32_t kFseWin = 16384;
struct FseDecWin {
    TableLdsT<kFblkLog> tab;
    DEntry dt[1u << kFblkLog];
    alignas(16) uint8_t win[kFseWin + 64];
};
struct FseDecLdsWin {
    FseDecWin w;
    int16_t norm[256];
    uint32_t tl;
    uint64_t hl;
    int32_t wb;  // the next window's first stream byte
    uint32_t done;
};
// Where the decode of fse_decode_run_lds stands: read position, the two states, symbols done.
struct FseDecPos {
    int32_t p;
    uint32_t s0, s1, i;
};
// fse_decode_run_lds over a window: win holds the stream bytes [wb, wb + kFseWin + 12) (wb a multiple
// of 4; bytes past the stream's end are not used). Decodes while the words of the next refill lie in
// the window, or to the end when the window starts at byte 0; returns whether all len symbols are
// done. first: the window holds the stream's end; take the start position and the two states.
__device__ __forceinline__ bool fse_decode_window(FseDecPos& z, const FZ_LDS DEntry* dt, const FZ_LDS uint8_t* win,
                                                  int32_t wb, bool first, uint64_t bsz, unsigned tl, uint8_t* out,
                                                  uint32_t len) {
    const FZ_LDS uint32_t* w32 = reinterpret_cast<const FZ_LDS uint32_t*>(win);
    const FZ_LDS uint32_t* dtw = reinterpret_cast<const FZ_LDS uint32_t*>(dt);
    uint64_t buf = 0;
    int32_t prel = 0;
    auto refill = [&]() {  // bits [p - 64, p); bytes below the start read as zero
        const int32_t lo = z.p - 64;
        const int32_t lc = max(lo, 0);
        const int32_t j0 = (lc >> 5) - (wb >> 2);
        const uint32_t sh = (uint32_t)lc & 31u;
        uint64_t b = (uint64_t)__builtin_amdgcn_alignbit(w32[j0 + 1], w32[j0], sh) |
                     ((uint64_t)__builtin_amdgcn_alignbit(w32[j0 + 2], w32[j0 + 1], sh) << 32);
        if (lo < 0) b = (z.p > 0 ? b << (uint32_t)(-lo) : 0ull);
        buf = b;
        prel = 64;
    };
    auto read = [&](uint32_t nb) -> uint32_t {
        prel -= (int32_t)nb;
        z.p -= (int32_t)nb;
        return (uint32_t)(buf >> ((uint32_t)prel & 63u)) & ((1u << nb) - 1u);
    };
    // How far the symbols can go before a refill would reach below the window: a refill needs
    // p - 64 >= 8 wb (or wb = 0), and a step of `step` symbols reads at most step * 11 bits, so
    // room / (step * 11) + 1 steps from here stay in the window (none when room < 0).
    auto limit = [&](uint32_t step) -> uint32_t {
        if (wb == 0) return len;
        const int32_t room = z.p - 64 - 8 * wb;
        if (room < 0) return z.i;
        const uint64_t k = (uint64_t)(room / (int32_t)(step * kFblkLog)) + 1;
        return (uint32_t)min<uint64_t>(len, z.i + step * k);
    };
    if (first) {
        z.p = (int32_t)((bsz - 1) * 8) + (int32_t)highbit32(win[bsz - 1 - (uint64_t)wb]);
        z.i = 0;
        refill();
        z.s0 = read(tl);
        z.s1 = read(tl);
    }
    while (z.i + 4 <= len) {
        const uint32_t lim = limit(4);
        if (z.i + 4 > lim) return false;
        for (; z.i + 4 <= lim; z.i += 4) {
            refill();
            const uint32_t e0 = dtw[z.s0], e1 = dtw[z.s1];
            z.s0 = (e0 & 0xFFFFu) + read(e0 >> 24);
            z.s1 = (e1 & 0xFFFFu) + read(e1 >> 24);
            const uint32_t f0 = dtw[z.s0], f1 = dtw[z.s1];
            z.s0 = (f0 & 0xFFFFu) + read(f0 >> 24);
            z.s1 = (f1 & 0xFFFFu) + read(f1 >> 24);
            const uint32_t v = ((e0 >> 16) & 0xFFu) | (((e1 >> 16) & 0xFFu) << 8) | (((f0 >> 16) & 0xFFu) << 16) |
                               (((f1 >> 16) & 0xFFu) << 24);
            *reinterpret_cast<uint32_t*>(out + z.i) = v;
        }
    }
    while (z.i + 2 <= len) {
        const uint32_t lim = limit(2);
        if (z.i + 2 > lim) return false;
        for (; z.i + 2 <= lim; z.i += 2) {
            refill();
            const uint32_t e0 = dtw[z.s0], e1 = dtw[z.s1];
            out[z.i] = (uint8_t)(e0 >> 16);
            out[z.i + 1] = (uint8_t)(e1 >> 16);
            z.s0 = (e0 & 0xFFFFu) + read(e0 >> 24);
            z.s1 = (e1 & 0xFFFFu) + read(e1 >> 24);
        }
    }
    if (z.i < len) out[z.i] = (uint8_t)(dtw[z.s0] >> 16);
    z.i = len;
    return true;
}

// Decodes framed class-byte blocks (the blocks of every stream of a call in one launch); the host
// found where each block starts.
// kBig: the layout of FseDecLds, for launches with a block whose table log is 12 or 13 (streams
// other encoders wrote); else FseDecLdsWin.
template <bool kBig>
__global__ void __launch_bounds__(256) k_fse_dec_blocks(const FseBlk* blks, int* err) {
    __shared__ std::conditional_t<kBig, FseDecLds, FseDecLdsWin> L;
    const FseBlk B = blks[blockIdx.x];
    const uint8_t* in = B.src;
    const uint32_t len = B.len;
    const uint8_t flag = in[0];
    uint8_t* dst = B.dst;
    if (flag == 0) {
        for (uint32_t i = threadIdx.x; i < len; i += blockDim.x) dst[i] = in[1 + i];
        return;
    }
    if (flag == 2) {
        for (uint32_t i = threadIdx.x; i < len; i += blockDim.x) dst[i] = in[1];
        return;
    }
    const uint8_t* src = in + 5;
    const uint32_t srcSize = (uint32_t)in[1] | ((uint32_t)in[2] << 8) | ((uint32_t)in[3] << 16) |
                             ((uint32_t)in[4] << 24);
    if (threadIdx.x == 0) {
        unsigned maxSym = 255, tl = 0;
        L.hl = read_ncount(L.norm, &maxSym, &tl, src, srcSize);
        for (unsigned s = maxSym + 1; s < 256; s++) L.norm[s] = 0;
        L.tl = tl;
    }
    __syncthreads();
    const uint64_t hl = L.hl;
    if (hl == kFseErr || hl >= srcSize) {
        if (threadIdx.x == 0) err[B.pad] = 1;
        return;
    }
    const unsigned tl = L.tl;
    const uint64_t bsz = srcSize - hl;
    if constexpr (!kBig) {
        if (tl > kFblkLog) {  // the host launches such blocks with the big layout
            if (threadIdx.x == 0) err[B.pad] = 1;
            return;
        }
        FseDecWin& W = L.w;
        const uint8_t* bs = src + hl;
        auto stage = [&](int32_t wb) {
            const uint64_t cnt = min<uint64_t>(kFseWin + 12, bsz - (uint64_t)wb);
            for (uint32_t u = threadIdx.x; u < cnt; u += blockDim.x) W.win[u] = bs[(uint64_t)wb + u];
        };
        W.tab.norm[threadIdx.x] = L.norm[threadIdx.x];
        int32_t wb = bsz > kFseWin ? (int32_t)((bsz - kFseWin) & ~(uint64_t)3) : 0;
        stage(wb);
        __syncthreads();
        if (!spread_parallel(W.tab, tl)) {
            if (threadIdx.x == 0) err[B.pad] = 1;
            return;
        }
        dtable_parallel(W.tab, tl, W.dt);
        __syncthreads();
        // lane 0 decodes a window at a time; between windows the workgroup stages the next one
        // (each lower than the last, the last one starting at byte 0)
        FseDecPos z{0, 0, 0, 0};
        for (bool first = true;; first = false) {
            if (threadIdx.x == 0) {
                bool fin;
                if (first && W.win[bsz - 1 - (uint64_t)wb] == 0) {
                    err[B.pad] = 1;
                    fin = true;
                } else {
                    fin = fse_decode_window(z, lds(W.dt), lds(W.win), wb, first, bsz, tl, dst, len);
                }
                const int32_t cur = max(z.p - 64, 0) >> 3;
                L.wb = cur > (int32_t)kFseWin - 16 ? (cur - ((int32_t)kFseWin - 16)) & ~3 : 0;
                L.done = fin ? 1u : 0u;
            }
            __syncthreads();
            if (L.done) return;
            wb = L.wb;
            stage(wb);
            __syncthreads();
        }
    } else {
        if (tl <= kFblkLog && bsz <= kFblk) {
            FseDecSmall& S = L.s;
            S.tab.norm[threadIdx.x] = L.norm[threadIdx.x];
            for (uint32_t i = threadIdx.x; i < bsz; i += blockDim.x) S.in[i] = src[hl + i];
            __syncthreads();
            if (!spread_parallel(S.tab, tl)) {
                if (threadIdx.x == 0) err[B.pad] = 1;
                return;
            }
            dtable_parallel(S.tab, tl, S.dt);
            __syncthreads();
            if (threadIdx.x == 0) {
                if (S.in[bsz - 1] == 0) err[B.pad] = 1;
                else fse_decode_run_lds(lds(S.dt), lds(S.in), bsz, tl, dst, len);
            }
            return;
        }
        FseDecBig& G = L.g;
        G.tab.norm[threadIdx.x] = L.norm[threadIdx.x];
        __syncthreads();
        if (!spread_parallel(G.tab, tl)) {
            if (threadIdx.x == 0) err[B.pad] = 1;
            return;
        }
        dtable_parallel(G.tab, tl, G.dt);
        __syncthreads();
        if (threadIdx.x != 0) return;
        if (src[hl + bsz - 1] == 0) {
            err[B.pad] = 1;
            return;
        }
        fse_decode_run(G.dt, src + hl, bsz, tl, dst, len);
    }
}

// ---------------------------------------------------------------- method 0 (RleFse:928-982)
struct NonZero {
    __device__ __forceinline__ bool operator()(int16_t c) const { return c != 0; }
};

__device__ inline int floor_log2_64(uint64_t v) { return 63 - __clzll((long long)v); }

// Run j precedes value j; the last run exists when the stream ends on the zero code.
__global__ void k_runs_values(const int16_t* bins, uint64_t n, const uint64_t* pos, uint64_t nv, uint64_t nr,
                              uint8_t* rcl, uint8_t* vcl, uint64_t* rbits, uint64_t* vbits) {
    const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < nr) {
        const uint64_t start = j ? pos[j - 1] + 1 : 0;
        const uint64_t end = j < nv ? pos[j] : n;
        const uint64_t L = end - start;
        const int k = floor_log2_64(L + 1);
        rcl[j] = (uint8_t)k;
        rbits[j] = (uint64_t)k;
    }
    if (j < nv) {
        const int32_t f = bins[pos[j]];
        const uint32_t zz = ((uint32_t)f << 1) ^ (uint32_t)(f >> 31);
        const int k = floor_log2_64((uint64_t)zz + 1);
        vcl[j] = (uint8_t)k;
        vbits[j] = (uint64_t)k;
    }
}

// MSB-first mantissa field (low k bits of v) at bit offset off of a big-endian bit string.
__device__ inline void put_msb_field(uint32_t* words, uint64_t off, uint64_t v, int k) {
    if (k <= 0) return;
    // bit p of the stream lives in byte p/8 at bit 7 - p%8; bytes map to little-endian words
    uint64_t bit = off;
    int left = k;
    while (left > 0) {
        const uint64_t byte = bit >> 3;
        const int inb = (int)(bit & 7);
        const int take = min(left, 8 - inb);
        const uint32_t chunk = (uint32_t)((v >> (left - take)) & ((1u << take) - 1));
        const uint32_t bits8 = chunk << (8 - inb - take);
        atomicOr(&words[byte >> 2], bits8 << (8 * (byte & 3)));
        left -= take;
        bit += take;
    }
}

__global__ void k_scatter_mantissas(const int16_t* bins, uint64_t n, const uint64_t* pos, uint64_t nv, uint64_t nr,
                                    const uint64_t* roff, const uint64_t* voff, const uint8_t* rcl, const uint8_t* vcl,
                                    uint32_t* rman, uint32_t* vman) {
    const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < nr) {
        const uint64_t start = j ? pos[j - 1] + 1 : 0;
        const uint64_t end = j < nv ? pos[j] : n;
        put_msb_field(rman, roff[j], end - start + 1, rcl[j]);
    }
    if (j < nv) {
        const int32_t f = bins[pos[j]];
        const uint32_t zz = ((uint32_t)f << 1) ^ (uint32_t)(f >> 31);
        put_msb_field(vman, voff[j], (uint64_t)zz + 1, vcl[j]);
    }
}

// ---------------------------------------------------------------- method 1 (RleFse:582-751)
struct IsO1Escape {
    __device__ __forceinline__ bool operator()(int16_t c) const { return o1_sym(c) == 255; }
};
struct CopyCode {
    const int16_t* codes;
    int16_t* out;
    __device__ __forceinline__ void operator()(uint64_t k, uint64_t i) const { out[k] = codes[i]; }
};

// Exact per-context histogram of a segment (N < 2^20): the context resets to that of 0 at each
// chunk start (RleFse:611-628).
__global__ void __launch_bounds__(256) k_o1_hist_exact(const int16_t* bins, uint64_t n, uint64_t cs, uint32_t* cnt) {
    __shared__ uint32_t h[kO1Ctx * kO1Sym];
    for (int i = threadIdx.x; i < kO1Ctx * kO1Sym; i += blockDim.x) h[i] = 0;
    __syncthreads();
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const int c = (i % cs == 0) ? 0 : o1_ctx(bins[i - 1]);
        atomicAdd(&h[c * kO1Sym + o1_sym(bins[i])], 1u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kO1Ctx * kO1Sym; i += blockDim.x)
        if (h[i]) atomicAdd(&cnt[i], h[i]);
}

// Windowed sample histogram (RleFse:641-658) of segment blockIdx.y (codes [g seg, g seg + seg) of the
// n): wlen-code windows every step = max(segment length / 2048, 512) codes, the context of each code
// taken from its true predecessor (0 at the segment start). The segments of a call in one launch. A
// workgroup takes every gridDim.x-th window: what a launch costs is the adds of its LDS counts to
// device memory, about 400 after one window and 2,500 after 30 (15 segments of 2,048 windows: 0.22 ms with
// a workgroup a window, under 0.08 with 1,024 workgroups).
__global__ void __launch_bounds__(256) k_o1_hist_sample(const int16_t* bins, uint64_t n, uint64_t seg, uint64_t wlen,
                                                        uint32_t* cnt) {
    __shared__ uint32_t h[kO1Ctx * kO1Sym];
    const uint64_t lo = (uint64_t)blockIdx.y * seg;
    bins += lo;
    cnt += (uint64_t)blockIdx.y * kO1Ctx * kO1Sym;
    n = min(seg, n - lo);
    const uint64_t step = max(n / 2048, (uint64_t)512);
    for (int i = threadIdx.x; i < kO1Ctx * kO1Sym; i += blockDim.x) h[i] = 0;
    __syncthreads();
    for (uint64_t w = (uint64_t)blockIdx.x * step; w < n; w += (uint64_t)gridDim.x * step) {
        const uint64_t we = min(w + wlen, n);
        for (uint64_t i = w + threadIdx.x; i < we; i += blockDim.x) {
            const int c = i ? o1_ctx(bins[i - 1]) : 0;
            atomicAdd(&h[c * kO1Sym + o1_sym(bins[i])], 1u);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kO1Ctx * kO1Sym; i += blockDim.x)
        if (h[i]) atomicAdd(&cnt[i], h[i]);
}

__global__ void k_add_one(uint32_t* cnt, int total) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < total) cnt[i] += 1;
}

// o1_normalize (RleFse:410-477): FSE_normalizeCount at tableLog 13, with the reference's fallback
// (proportional counts, surplus to the largest, deficit taken from the largest ones) when it fails
// or when a context has at most one symbol. h and f are in LDS; f receives the counts. The first part
// of FSE_normalizeCount runs with a thread per symbol; where its rounding leaves too much to give to
// the largest count (its second method), and for the fallback, one lane does all of it.
struct O1NormLds {
    uint32_t h[kO1Sym];
    int16_t norm[kO1Sym];
    uint64_t part[4];
    uint32_t best;
    int sum;
};
__device__ void o1_normalize_lane(O1NormLds& L, uint64_t total, int nonzero) {
    const uint32_t* h = L.h;
    int16_t* f = L.norm;
    const int M = 1 << kO1Log;
    if (nonzero > 1 && normalize_count(f, kO1Log, h, total, kO1Sym - 1) != kFseErr) return;
    int sum = 0, maxf = 0, argmax = 0;
    for (int s = 0; s < kO1Sym; s++) {
        if (h[s]) {
            int v = (int)((uint64_t)h[s] * (uint64_t)M / total);
            if (v == 0) v = 1;
            f[s] = (int16_t)v;
            sum += v;
            if (v > maxf) { maxf = v; argmax = s; }
        } else {
            f[s] = 0;
        }
    }
    int e = M - sum;
    if (e > 0) {
        f[argmax] = (int16_t)(f[argmax] + e);
    } else if (e < 0) {
        e = -e;
        int take = (maxf - 1 < e) ? (maxf - 1) : e;
        f[argmax] = (int16_t)(f[argmax] - take);
        e -= take;
        while (e > 0) {
            int mi = -1;
            uint32_t mv = 1;
            for (int s = 0; s < kO1Sym; s++)
                if ((uint16_t)f[s] > mv) { mv = (uint16_t)f[s]; mi = s; }
            if (mi < 0) break;
            take = (int)(uint16_t)f[mi] - 1;
            if (take > e) take = e;
            f[mi] = (int16_t)(f[mi] - take);
            e -= take;
        }
    }
}
// by the 256 threads of a workgroup, L.h set
__device__ void o1_normalize(O1NormLds& L) {
    const unsigned t = threadIdx.x;
    const uint32_t c = L.h[t];
    uint64_t sum;
    block_scan_u64((uint64_t)c | (uint64_t)(c != 0) << 48, L.part, &sum);
    const uint64_t total = sum & ((1ull << 48) - 1);
    const int nonzero = (int)(sum >> 48);
    if (total == 0) {
        L.norm[t] = t == 0 ? (int16_t)(1 << kO1Log) : (int16_t)0;
        __syncthreads();
        return;
    }
    if (t == 0) {
        L.best = 0;
        L.sum = 0;
    }
    __syncthreads();
    bool whole = nonzero > 1 && kO1Log >= min_table_log(total, kO1Sym - 1);
    if (whole) {
        const uint32_t rtb[8] = {0, 473195, 504333, 520860, 550000, 700000, 750000, 830000};
        const uint64_t scale = 62 - kO1Log, step = ((uint64_t)1 << 62) / total, vStep = 1ull << (scale - 20);
        int16_t p = 0;
        int used = 0;
        if (c != 0 && c <= (uint32_t)(total >> kO1Log)) {
            p = -1;
            used = 1;
        } else if (c != 0) {
            const uint64_t scaled = (uint64_t)c * step;
            p = (int16_t)(scaled >> scale);
            if (p < 8) p = (int16_t)(p + ((scaled - ((uint64_t)p << scale)) > vStep * rtb[p]));
            used = p;
            // the largest count, the first of equal ones
            if (p > 0) atomicMax(&L.best, (uint32_t)p << 16 | (255u - t));
        }
        L.norm[t] = p;
        if (used) atomicAdd(&L.sum, used);
        __syncthreads();
        const unsigned largest = L.best ? 255u - (L.best & 0xFFFFu) : 0u;
        const int still = (1 << kO1Log) - L.sum;
        const int lp = L.norm[largest];
        __syncthreads();
        whole = !(-still >= (lp >> 1));
        if (whole && t == largest) L.norm[t] = (int16_t)(lp + still);
    }
    if (!whole && t == 0) o1_normalize_lane(L, total, nonzero);
    __syncthreads();
}

// Encoding tables of every context of every segment: grid (contexts, segments).
__global__ void __launch_bounds__(256) k_o1_tables(const uint32_t* cnt_all, uint16_t* nf_all, CTable* ct_all, uint32_t* use) {
    __shared__ TableLds L;
    __shared__ O1NormLds N;
    __shared__ uint32_t sum;
    const unsigned t = threadIdx.x;
    const size_t c = (size_t)blockIdx.y * kO1Ctx + blockIdx.x;
    if (t == 0) sum = 0;
    __syncthreads();
    uint32_t h = cnt_all[c * kO1Sym + t];
    N.h[t] = h;
#pragma unroll
    for (int d = 32; d; d >>= 1) h += __shfl_xor(h, d, 64);
    if ((t & 63u) == 0) atomicAdd(&sum, h);
    __syncthreads();
    if (t == 0) use[c] = sum;
    o1_normalize(N);
    nf_all[c * kO1Sym + t] = (uint16_t)N.norm[t];
    L.norm[t] = N.norm[t];
    __syncthreads();
    if (!spread_parallel(L, kO1Log)) return;  // cannot happen for counts from o1_normalize
    ctable_parallel(L, kO1Log, kO1Sym - 1, ct_all + c);
}


// ---- order-1 tANS encoding split into pieces --------------------------------------------------
// A chain is encoded backwards: symbol hi-1 seeds the state (FSE_initCState2), then one encoder
// step per symbol i = hi-2 .. lo. The steps are cut into pieces of consecutive steps,
// piece 0 holding the first steps (i = hi-2 downwards). A piece's output bits depend on the state
// it starts from, which the previous piece produces. Encoder steps are many-to-one (the low bits
// of the state leave through the bitstream), so runs from different start states merge, all but
// a handful within a hundred steps and the last few within thousands. Every piece emits its bits at its
// offset in the chain (k_o1_emit) once its start state is known, which is found in one of two ways;
// the result is the sequential encoder's bitstream either way.
// - Arrays of up to kSetMaxCodes codes, where a step's latency (its table is read from L2: 0.35 us with a
//   state of its own in every lane, 0.13 us with a few) is all that counts: a wave a piece of kSetPiece steps follows every state that can enter the piece
//   (k_o1_sets), and a walk over the pieces picks the true ones (k_o1_sets_walk).
// - Longer arrays fill the chip with one lane a piece of kO1Piece steps: all run from a guessed state
//   (k_o1_spec), then each re-runs from its predecessor's end state until it meets its own logged
//   trajectory (k_o1_fix, repeated while some piece fails to meet it).
// 540,000 codes, the order-1 stage without its side streams: guessed and repaired 1.4 to 6 ms (2 to 10
// rounds, as slowly as the last states merge), by sets 0.25 ms; 86,000: 1.03 and 0.24 ms. By sets a
// code costs 2.25 steps of a wave: 134 million codes, 1.3 ms guessed, repaired and emitted, would take 7.
constexpr uint32_t kO1Piece = 1024, kO1PieceMin = 256;  // as many pieces as the chip has lanes in one round of workgroups
constexpr uint32_t kEncThreads = 1024, kEmitThreads = 1024, kRingWords = 8;
constexpr int kEncHot = 8, kEmitHot = 6;  // state tables in LDS: 158 KB with the per-symbol arrays (and the emit's rings)
constexpr uint32_t kSetPiece = 256;
constexpr uint64_t kSetMaxCodes = 7ull << 19;  // 3,584 pieces a chain: the walk's links fit 64 KB of LDS
constexpr uint32_t kSetStates = 16;    // states followed through a piece
constexpr uint32_t kSetWarm = 320;     // steps in front of a piece; the first 128 are searched for a rare symbol
constexpr uint32_t kSetSearch = 128;
constexpr uint32_t kSetWarmMax = 1344; // how far back the search goes

struct O1Chains {        // device view of the chains of one call
    const uint64_t* c;   // 4 per chain: segment lo, chunk lo, chunk hi, segment
    const uint64_t* pfirst;  // first piece of each chain (exclusive scan), nchains + 1 entries
    int nchains;
    uint32_t piece;          // steps of a piece
};

__device__ inline int o1_piece_chain(const O1Chains& C, uint64_t pid) {
    int lo = 0, hi = C.nchains;  // last chain with pfirst <= pid
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (C.pfirst[mid] <= pid) lo = mid; else hi = mid;
    }
    return lo;
}

// Steps [s_hi down to s_lo] of piece p of a chain with symbols [lo, hi): s_hi = hi-2 - p*piece.
__device__ inline void o1_piece_range(uint32_t piece, uint64_t lo, uint64_t hi, uint64_t p, uint64_t& s_hi, uint64_t& s_lo) {
    s_hi = hi - 2 - p * piece;
    s_lo = (s_hi + 1 > lo + piece) ? s_hi + 1 - piece : lo;
}

__device__ inline uint32_t o1_seed_state(const int16_t* bins, uint64_t lo, uint64_t idx, const CTable* ct) {
    const int prev = (idx > lo) ? bins[idx - 1] : 0;
    return init_state2(&ct[o1_ctx(prev)], o1_sym(bins[idx]));
}

// One segment's encoding tables in LDS: the per-symbol arrays of all 15 contexts, and the state tables
// (16 KB each) of the H contexts that occur most often. With the state tables in L2 the lanes of a
// full chip wait for its rate of requests (a lane reads one entry a step from anywhere in 240 KB: 160 G
// steps/s); with 8 of them in LDS a step waits for L2 only in the waves that hold a rare context, and
// its instructions count as much. 134 million codes of a k^-3 field, REL 1e-3 (one in 2,700 an escape): k_o1_spec
// 0.84 -> 0.36 ms, k_o1_fix 0.92 -> 0.49, k_o1_emit (6 tables, the rings beside them) 0.97 -> 0.45; 1e-4 (one in two):
// 1.09 -> 0.39, 2.84 -> 2.38 (beside the escapes' blocks, which come at once now), 1.41 -> 0.41.
template <int H>
struct O1EncLds {
    // a symbol's deltaNbBits, and its deltaFindState + 8,192 * place of the context's state table: below H
    // in st, else H + context
    u32x2 sym[kO1Ctx * kO1Sym];
    uint16_t st[(size_t)H << kO1Log];
    uint32_t place[kO1Ctx + 1];
};
template <int H>
struct O1EncTab {
    const FZ_LDS u32x2* sym;
    const FZ_LDS uint16_t* st;
    const FZ_GLB uint16_t* far;
};
// Stages the tables of segment seg. Every thread of the workgroup calls it.
template <int H>
__device__ inline O1EncTab<H> o1_stage_tables(O1EncLds<H>& T, const CTable* ct, const uint32_t* use) {
    if (threadIdx.x < kO1Ctx) {
        const uint32_t c = threadIdx.x, u = use[c];
        uint32_t rank = 0;
        for (uint32_t j = 0; j < (uint32_t)kO1Ctx; j++) rank += use[j] > u || (use[j] == u && j < c) ? 1u : 0u;
        T.place[c] = rank < (uint32_t)H ? rank : (uint32_t)H + c;
    }
    __syncthreads();
    for (uint32_t u = threadIdx.x; u < kO1Ctx * kO1Sym; u += blockDim.x) {
        T.sym[u] = u32x2{ct[u / kO1Sym].deltaNbBits[u % kO1Sym],
                         (uint32_t)ct[u / kO1Sym].deltaFindState[u % kO1Sym] + (T.place[u / kO1Sym] << kO1Log)};
    }
    for (uint32_t c = 0; c < (uint32_t)kO1Ctx; c++) {
        if (T.place[c] >= (uint32_t)H) continue;
        const uint32_t* from = reinterpret_cast<const uint32_t*>(ct[c].stateTable);
        uint32_t* to = reinterpret_cast<uint32_t*>(T.st + (T.place[c] << kO1Log));
        for (uint32_t i = threadIdx.x; i < 1u << (kO1Log - 1); i += blockDim.x) to[i] = from[i];
    }
    __syncthreads();
    return O1EncTab<H>{lds(T.sym), lds(T.st),
                       glb(reinterpret_cast<const uint16_t*>(ct)) + offsetof(CTable, stateTable) / 2};
}
// o1_ctx(prev) * 256 + o1_sym(code) in a few instructions: the context of a magnitude up to 12 is a nibble.
__device__ __forceinline__ uint32_t o1_index(int code, int prev) {
    const uint32_t a = min((uint32_t)(prev < 0 ? -prev : prev), 12u);
    const uint32_t cx = ((uint32_t)(0xDBBBB99975310ull >> (4 * a)) & 15u) + ((uint32_t)prev >> 31);
    return cx * kO1Sym + min(((uint32_t)code << 1) ^ (uint32_t)(code >> 31), 255u);
}
__host__ __device__ constexpr bool o1_index_holds() {
    for (int v = 0; v < 40; v++) {
        const int m = v <= 4 ? v - 1 : v <= 7 ? 4 : v <= 11 ? 5 : 6;
        if ((int)(0xDBBBB99975310ull >> (4 * (v < 12 ? v : 12)) & 15u) != (v ? 1 + 2 * m : 0)) return false;
    }
    return true;
}
static_assert(o1_index_holds(), "the nibbles are o1_ctx");

// The bits that a step of symbol d emits from a state, and the state after it.
__device__ __forceinline__ uint32_t o1_step_bits(uint32_t state, u32x2 d) { return (state + d.x) >> 16; }
template <int H>
__device__ __forceinline__ uint32_t o1_step_next(const O1EncTab<H>& T, uint32_t state, u32x2 d, uint32_t bits) {
    constexpr uint32_t kNear = (uint32_t)H << kO1Log;
    const uint32_t at = (state >> bits) + d.y;
    uint32_t v = T.st[min(at, kNear - 1)];
    if (at >= kNear) {
        const uint32_t j = at - kNear;
        v = T.far[(j >> kO1Log) * (uint32_t)(sizeof(CTable) / 2) + (j & ((1u << kO1Log) - 1u))];
    }
    return v;
}

// The lane's piece in a launch of whole workgroups a segment (every workgroup's pieces share the tables
// that it stages); ~0 past the segment's last piece. seg: the workgroup's segment.
__device__ __forceinline__ uint64_t o1_piece_of(const O1Chains& C, uint32_t groups, uint32_t& seg) {
    const uint32_t b = xcd_block();
    seg = b / groups;
    const uint64_t pid = C.pfirst[seg * kO1K] + (uint64_t)(b % groups) * blockDim.x + threadIdx.x;
    return pid < C.pfirst[(seg + 1) * kO1K] ? pid : ~0ull;
}

// Runs step(u, k) for the steps i = 8c + k from s_hi down to s_lo of a piece, u the step's o1_index
// (previous code 0 at the chain's first symbol lo), begin(8c) before and more() after those of a group of
// eight; ends early when more returns false. A lane's codes come 32 at a time in four 16-byte loads of
// the same 64 bytes, the next 32 in flight: the open lines of a full chip's lanes (one each, 33 MB) do not
// stay in L2, and eight loads a line fetched the codes five times (k_o1_spec 0.40 ms, k_o1_emit 0.50; 0.37 and 0.45 so). A step costs its instructions as much
// as its waits (16 waves a CU), so blocks of 32 inside the piece, nearly all, run without tests of their
// bounds. bins is 16-byte aligned and its allocation extends to the next multiple of 16 bytes.
template <typename B, typename F, typename M>
__device__ __forceinline__ void o1_piece_codes(const int16_t* bins, uint64_t lo, uint64_t s_hi, uint64_t s_lo, B&& begin,
                                               F&& step, M&& more) {
    const u32x4* b4 = reinterpret_cast<const u32x4*>(bins);
    // v[k + 1]: code k of a group of eight; v[0]: the code in front of it
    auto codes = [](u32x4 w, u32x4 before, int (&v)[9]) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
            v[2 * k + 1] = (int)(int16_t)(w[k] & 0xFFFFu);
            v[2 * k + 2] = (int)w[k] >> 16;
        }
        v[0] = (int)before[3] >> 16;
    };
    const u32x4 zero{0u, 0u, 0u, 0u};
    u32x4 cur[4] = {zero, zero, zero, zero}, nxt[4] = {zero, zero, zero, zero};
    uint64_t blk = s_hi >> 5;
    const uint64_t blk_lo = s_lo >> 5;
    auto inside = [&](uint64_t k) { return 32 * k >= s_lo && 32 * k + 31 <= s_hi && 32 * k > lo; };
    if (inside(blk)) {
#pragma unroll
        for (int g = 0; g < 4; g++) cur[g] = b4[4 * blk + g];
    }
    for (;;) {
        if (blk > 0) {
#pragma unroll
            for (int g = 0; g < 4; g++) nxt[g] = b4[4 * (blk - 1) + g];
        }
        int v[9];
        if (inside(blk)) {
#pragma unroll
            for (int g = 3; g >= 0; g--) {
                begin(32 * blk + 8 * g);
                codes(cur[g], g > 0 ? cur[g - 1] : nxt[3], v);
#pragma unroll
                for (int k = 7; k >= 0; k--) step(o1_index(v[k + 1], v[k]), k);
                if (!more()) return;
            }
        } else {
            for (int g = 3; g >= 0; g--) {
                const uint64_t c = 4 * blk + g, base = 8 * c;
                if (base > s_hi || base + 7 < s_lo) continue;
                begin(base);
                codes(b4[c], c > 0 ? b4[c - 1] : zero, v);
#pragma unroll
                for (int k = 7; k >= 0; k--) {
                    const uint64_t i = base + (uint64_t)k;
                    if (i <= s_hi && i >= s_lo) step(o1_index(v[k + 1], i > lo ? v[k] : 0), k);
                }
                if (!more()) return;
            }
        }
        if (blk == blk_lo) return;
        blk--;
#pragma unroll
        for (int g = 0; g < 4; g++) cur[g] = nxt[g];
    }
}
struct PieceNoop {
    __device__ __forceinline__ void operator()(uint64_t) const {}
    __device__ __forceinline__ bool operator()() const { return true; }
};

__global__ void __launch_bounds__(kEncThreads) k_o1_spec(const int16_t* bins, O1Chains C, uint32_t groups, uint64_t npieces,
                                                         const CTable* ct_all, const uint32_t* use, uint16_t* slog,
                                                         uint32_t* end_state, uint64_t* nbits) {
    __shared__ O1EncLds<kEncHot> L;
    uint32_t seg;
    const uint64_t pid = o1_piece_of(C, groups, seg);
    const CTable* ct = ct_all + (size_t)seg * kO1Ctx;
    const auto T = o1_stage_tables(L, ct, use + seg * kO1Ctx);
    if (pid == ~0ull) return;
    const int q = o1_piece_chain(C, pid);
    const uint64_t lo = C.c[4 * q + 1], hi = C.c[4 * q + 2];
    const uint64_t p = pid - C.pfirst[q];
    uint64_t s_hi, s_lo;
    o1_piece_range(C.piece, lo, hi, p, s_hi, s_lo);
    // piece 0 starts from the true seed; the others from the seed their own first symbol would give
    uint32_t st = o1_seed_state(bins, lo, p == 0 ? hi - 1 : s_hi, ct);
    uint32_t bits = 0;
    // the log is step-major (step j of every piece side by side), so a wave's writes are coalesced
    uint16_t* log = slog + pid;
    o1_piece_codes(bins, lo, s_hi, s_lo, PieceNoop{}, [&](uint32_t u, int) {
        *log = (uint16_t)st;
        log += npieces;
        const u32x2 d = T.sym[u];
        const uint32_t nb = o1_step_bits(st, d);
        bits += nb;
        st = o1_step_next(T, st, d, nb);
    }, PieceNoop{});
    end_state[pid] = st;
    nbits[pid] = bits;
}

// One fix-up round over the end states of the previous round (end_prev, spec_end in the first).
// A piece whose predecessor ended differently in the previous round (every piece in the first
// round) re-runs from that end state until its state equals its logged one; from there on its bits
// and end state are those of its logged run. One that never meets its log ends in the state its
// re-run reached. A piece whose end state differs from end_prev marks itself changed, and its
// successor runs again in the next round; after a round with no change every piece started from
// its predecessor's true end state. Piece 0 of a chain starts from the true seed and never changes.
__global__ void __launch_bounds__(kEncThreads) k_o1_fix(const int16_t* bins, O1Chains C, uint32_t groups, uint64_t npieces,
                                                const CTable* ct_all, const uint32_t* use, const uint16_t* slog,
                                                const uint32_t* spec_end,
                                                const uint64_t* spec_bits, const uint32_t* end_prev,
                                                uint32_t* end_next, uint64_t* nbits, const uint8_t* changed_prev,
                                                uint8_t* changed_next, unsigned int* any_changed) {
    __shared__ O1EncLds<kEncHot> L;
    uint32_t seg;
    const uint64_t pid = o1_piece_of(C, groups, seg);
    int q = 0;
    uint64_t p = 0;
    bool again = false;
    if (pid != ~0ull) {
        q = o1_piece_chain(C, pid);
        p = pid - C.pfirst[q];
        again = p > 0 && (changed_prev == nullptr || changed_prev[pid - 1]);
    }
    O1EncTab<kEncHot> T{};
    // the tables are staged where a lane needs them: after the first rounds that is in few workgroups
    if (__syncthreads_or(again)) T = o1_stage_tables(L, ct_all + (size_t)seg * kO1Ctx, use + seg * kO1Ctx);
    if (pid == ~0ull) return;
    uint32_t end = end_prev[pid];
    uint8_t ch = 0;
    if (again) {
        const uint64_t lo = C.c[4 * q + 1], hi = C.c[4 * q + 2];
        uint64_t s_hi, s_lo;
        o1_piece_range(C.piece, lo, hi, p, s_hi, s_lo);
        uint32_t st = end_prev[pid - 1];
        int32_t delta = 0;
        bool met = false;
        // The logged states of eight steps come together: a load a step would double a step's time, and
        // the few lanes that are long without meeting their log decide a round's. After the states have
        // met they stay together, so that the rest of the eight steps changes nothing.
        uint32_t log8[8];
        o1_piece_codes(bins, lo, s_hi, s_lo, [&](uint64_t base) {
#pragma unroll
            for (int k = 0; k < 8; k++)
                log8[k] = slog[(s_hi - min(max(base + (uint64_t)k, s_lo), s_hi)) * npieces + pid];
        }, [&](uint32_t u, int k) {
            met = met || st == log8[k];
            const u32x2 d = T.sym[u];
            const uint32_t nb = o1_step_bits(st, d);
            delta += (int32_t)nb - (int32_t)o1_step_bits(log8[k], d);
            st = o1_step_next(T, st, d, nb);
        }, [&]() { return !met; });
        nbits[pid] = (uint64_t)((int64_t)spec_bits[pid] + delta);
        const uint32_t e = met ? spec_end[pid] : st;
        if (e != end) {
            end = e;
            ch = 1;
            atomicAdd(any_changed, 1u);
        }
    }
    end_next[pid] = end;
    changed_next[pid] = ch;
}

// Chain-relative bit offset of every piece and the bit count of every chain's steps, from the
// exclusive scan of the piece bit counts over all pieces.
__global__ void __launch_bounds__(256) k_o1_offsets(O1Chains C, uint64_t npieces, const uint64_t* scan,
                                                    const uint64_t* nbits, uint64_t* bitoff, uint64_t* chain_bits) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < npieces) {
        const int q = o1_piece_chain(C, t);
        bitoff[t] = scan[t] - scan[C.pfirst[q]];
    } else if (t < npieces + (uint64_t)C.nchains) {
        const uint64_t q = t - npieces;
        const uint64_t a = C.pfirst[q], b = C.pfirst[q + 1];
        chain_bits[q] = (b > a) ? scan[b - 1] + nbits[b - 1] - scan[a] : 0;
    }
}

// Clears the 32-bit words that several pieces share (each piece's first word, and the words of the
// chain's closing bits); every other word of a chain is written whole by exactly one piece.
__global__ void __launch_bounds__(256) k_o1_clear_shared(O1Chains C, uint64_t npieces, const uint64_t* bitoff,
                                                         const uint64_t* chain_bits, uint32_t* words,
                                                         uint64_t stride_words) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < npieces) {
        const int q = o1_piece_chain(C, t);
        words[q * stride_words + (bitoff[t] >> 5)] = 0;
    } else if (t < npieces + (uint64_t)C.nchains) {
        const uint64_t q = t - npieces;
        const uint64_t b = chain_bits[q];  // bits before the closing state
        for (uint64_t w = b >> 5; w <= (b + kO1Log + 1) >> 5; w++) words[q * stride_words + w] = 0;
    }
}

struct WordWriter {  // LSB-first bits into 32-bit words; shared (first and last) words are OR-ed in
    uint32_t* w;
    uint64_t idx;
    uint64_t acc;
    uint32_t n;
    bool first;
};
__device__ inline void ww_put(WordWriter& W, uint32_t v, uint32_t nb) {
    if (!nb) return;
    W.acc |= (uint64_t)(v & ((1u << nb) - 1)) << W.n;
    W.n += nb;
    if (W.n >= 32) {
        if (W.first) { atomicOr(&W.w[W.idx], (uint32_t)W.acc); W.first = false; }
        else W.w[W.idx] = (uint32_t)W.acc;
        W.idx++;
        W.acc >>= 32;
        W.n -= 32;
    }
}
// k_o1_emit's output: a lane's words pass through an 8-word LDS ring and leave in aligned 32-byte
// runs (the lanes of a wave write 131 K pieces' lines at once, and single-word stores leave partly
// written lines to L2 evictions). The first word (shared with the previous piece) is OR-ed in; the
// words before the first 32-byte boundary, and those after the last full run, go one by one; the last,
// partial word (shared with the next piece) is OR-ed in.
struct RunWriter {
    uint32_t* w;            // the chain's words
    FZ_LDS uint32_t* ring;  // this lane's kRingWords words
    uint64_t idx;           // the word being filled
    uint64_t acc;
    uint32_t n;
    bool first, runs;       // runs: a 32-byte boundary has been passed
};
__device__ inline void rw_word(RunWriter& W, uint32_t v) {
    if (W.first) {
        atomicOr(&W.w[W.idx], v);
        W.first = false;
    } else if (!W.runs) {
        W.w[W.idx] = v;
    } else {
        W.ring[W.idx & (kRingWords - 1)] = v;
        if ((W.idx & (kRingWords - 1)) == kRingWords - 1) {
            const FZ_LDS u32x4* r = reinterpret_cast<const FZ_LDS u32x4*>(W.ring);
            u32x4* d = reinterpret_cast<u32x4*>(W.w + (W.idx - (kRingWords - 1)));
            const u32x4 r0 = r[0], r1 = r[1];
            d[0] = r0;
            d[1] = r1;
        }
    }
    W.idx++;
    if ((W.idx & (kRingWords - 1)) == 0) W.runs = true;
}
__device__ inline void rw_put(RunWriter& W, uint32_t v, uint32_t nb) {
    if (!nb) return;
    W.acc |= (uint64_t)(v & ((1u << nb) - 1)) << W.n;
    W.n += nb;
    if (W.n >= 32) {
        rw_word(W, (uint32_t)W.acc);
        W.acc >>= 32;
        W.n -= 32;
    }
}
__device__ inline void rw_flush(RunWriter& W) {
    if (W.runs)
        for (uint64_t k = W.idx & ~(uint64_t)(kRingWords - 1); k < W.idx; k++) W.w[k] = W.ring[k & (kRingWords - 1)];
    if (W.n) atomicOr(&W.w[W.idx], (uint32_t)W.acc);
}

__global__ void __launch_bounds__(kEmitThreads) k_o1_emit(const int16_t* bins, O1Chains C, uint32_t groups,
                                                          const CTable* ct_all, const uint32_t* use,
                                                          const uint32_t* end_state, const uint64_t* bitoff,
                                                          uint32_t* words, uint64_t stride_words, const uint64_t* failed) {
    __shared__ O1EncLds<kEmitHot> L;
    __shared__ __align__(16) uint32_t ring[kEmitThreads * kRingWords];
    if (failed && *failed) return;
    uint32_t seg;
    const uint64_t pid = o1_piece_of(C, groups, seg);
    const CTable* ct = ct_all + (size_t)seg * kO1Ctx;
    const auto T = o1_stage_tables(L, ct, use + seg * kO1Ctx);
    if (pid == ~0ull) return;
    const int q = o1_piece_chain(C, pid);
    const uint64_t lo = C.c[4 * q + 1], hi = C.c[4 * q + 2];
    const uint64_t p = pid - C.pfirst[q];
    uint64_t s_hi, s_lo;
    o1_piece_range(C.piece, lo, hi, p, s_hi, s_lo);
    uint32_t st = p == 0 ? o1_seed_state(bins, lo, hi - 1, ct) : end_state[pid - 1];
    const uint64_t b0 = bitoff[pid];
    RunWriter W{words + q * stride_words, lds(ring + threadIdx.x * kRingWords), b0 >> 5, 0, (uint32_t)(b0 & 31), true, false};
    o1_piece_codes(bins, lo, s_hi, s_lo, PieceNoop{}, [&](uint32_t u, int) {
        const u32x2 d = T.sym[u];
        const uint32_t nb = o1_step_bits(st, d);
        rw_put(W, st, nb);
        st = o1_step_next(T, st, d, nb);
    }, PieceNoop{});
    rw_flush(W);
}

// The states that can enter a piece and what becomes of them: kSetStates slots a piece.
struct O1Sets {
    uint16_t *start, *end, *bits;
    uint8_t* cnt;  // slots in use
};

// Steps hi_i down to lo_i for the state of every lane: the lanes read and look up 64 steps at once
// (their symbols do not depend on the states), the next 64 in flight; a step then takes its two
// numbers from the lane that holds them.
__device__ __forceinline__ void o1_set_run(const int16_t* bins, uint64_t lo, uint64_t hi_i, uint64_t lo_i,
                                           const CTable* ct, uint32_t& st, uint32_t& bits) {
    if (hi_i < lo_i) return;
    const uint32_t lane = threadIdx.x & 63u;
    const FZ_GLB uint16_t* tab = glb(reinterpret_cast<const uint16_t*>(ct));
    auto load = [&](uint64_t top, uint32_t& d, uint32_t& b) {
        const uint64_t i = top >= lo_i + lane ? top - lane : lo_i;
        const int cx = o1_ctx(i > lo ? bins[i - 1] : 0), sym = o1_sym(bins[i]);
        d = ct[cx].deltaNbBits[sym];
        b = (uint32_t)(cx * (sizeof(CTable) / 2) + offsetof(CTable, stateTable) / 2) + (uint32_t)ct[cx].deltaFindState[sym];
    };
    uint32_t d, b, dn, bn;
    load(hi_i, dn, bn);
    const uint64_t steps = hi_i - lo_i + 1;
    for (uint64_t done = 0; done < steps; done += 64) {
        d = dn;
        b = bn;
        if (done + 64 < steps) load(hi_i - done - 64, dn, bn);
        auto step = [&](int k) {
            const uint32_t nb = (st + (uint32_t)__builtin_amdgcn_readlane((int)d, k)) >> 16;
            bits += nb;
            st = tab[(st >> nb) + (uint32_t)__builtin_amdgcn_readlane((int)b, k)];
        };
        const int cnt = (int)min(steps - done, (uint64_t)64);
        if (cnt == 64) {
#pragma unroll 16
            for (int k = 0; k < 64; k++) step(k);
        } else {
            for (int k = 0; k < cnt; k++) step(k);
        }
    }
}

// A wave a piece. After a step whose symbol has the normalized count c, only c of the 8,192 states are
// left, whatever the state before: the symbol of the lowest count among 128 some way in front of the piece
// gives the first set, one state a lane (a symbol of a count up to 64; none there, the search goes on
// further back). On the way to the piece most of them merge: 5 are left in the median over fields at
// bounds 1e-2 to 1e-4, at most 8 seen. failed: a piece without such a symbol, or with more than kSetStates
// states left. Bound by the latency of the steps' table reads.
__global__ void __launch_bounds__(256) k_o1_sets(const int16_t* bins, O1Chains C, uint64_t npieces, const CTable* ct_all,
                                                 const uint16_t* nf, O1Sets B, uint64_t* failed) {
    const uint32_t lane = threadIdx.x & 63u;
    const uint64_t pid = uniform32((uint32_t)(xcd_block() * 4u + (threadIdx.x >> 6)));
    if (pid >= npieces) return;
    const int q = o1_piece_chain(C, pid);
    const uint64_t lo = uniform64(C.c[4 * q + 1]), hi = uniform64(C.c[4 * q + 2]), seg = uniform64(C.c[4 * q + 3]);
    const CTable* ct = ct_all + seg * kO1Ctx;
    const uint16_t* norm = nf + seg * kO1Ctx * kO1Sym;
    uint64_t s_hi, s_lo;
    o1_piece_range(C.piece, lo, hi, pid - uniform64(C.pfirst[q]), s_hi, s_lo);
    uint32_t st, bits = 0;
    uint64_t from = hi - 1;  // the step before the first one run
    uint32_t states = 1;
    bool exact = true;
    for (uint64_t warm = kSetWarm; s_hi + warm < hi - 1; warm += kSetSearch) {
        // steps s_hi + warm downwards
        uint32_t best = ~0u;
#pragma unroll
        for (uint32_t h = 0; h < kSetSearch; h += 64) {
            const uint64_t i = s_hi + warm - h - lane;  // above s_lo: kSetWarm > kSetSearch
            const uint32_t c = norm[o1_ctx(bins[i - 1]) * kO1Sym + o1_sym(bins[i])];
            const uint32_t cc = c == 0xFFFFu ? 1u : c == 0 ? 0xFFFFu : c;  // -1 stands for 1
            best = min(best, cc << 8 | (h + lane));
        }
#pragma unroll
        for (uint32_t d = 32; d; d >>= 1) best = min(best, (uint32_t)__shfl_xor((int)best, (int)d, 64));
        best = uniform32(best);
        if (best >> 8 <= 64) {
            exact = false;
            from = s_hi + warm - (best & 255u);
            states = best >> 8;
            break;
        }
        if (warm + kSetSearch > kSetWarmMax) {
            if (lane == 0) atomicOr(reinterpret_cast<unsigned long long*>(failed), 1ull);
            return;
        }
    }
    if (exact) {
        st = o1_seed_state(bins, lo, hi - 1, ct);
    } else {
        const CTable& t = ct[o1_ctx(bins[from - 1])];
        st = t.stateTable[t.deltaFindState[o1_sym(bins[from])] + (int32_t)(states + min(lane, states - 1))];
    }
    o1_set_run(bins, lo, from - 1, s_hi + 1, ct, st, bits);
    // one slot for each state that is left
    uint32_t cnt = 0, slot_state = uniform32(st);
    for (uint64_t left = __ballot(1); left; cnt++) {
        const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)st, __ffsll((unsigned long long)left) - 1);
        left &= ~__ballot(st == v);
        if (lane == cnt) slot_state = v;
    }
    if (cnt > kSetStates) {
        if (lane == 0) atomicOr(reinterpret_cast<unsigned long long*>(failed), 1ull);
        return;
    }
    st = slot_state;
    bits = 0;
    if (lane < kSetStates) B.start[pid * kSetStates + lane] = lane < cnt ? (uint16_t)st : (uint16_t)0;
    if (lane == 0) B.cnt[pid] = (uint8_t)cnt;
    o1_set_run(bins, lo, s_hi, s_lo, ct, st, bits);
    if (lane < cnt) {
        B.end[pid * kSetStates + lane] = (uint16_t)st;
        B.bits[pid * kSetStates + lane] = (uint16_t)bits;
    }
}

// One workgroup a chain: every slot's end among the next piece's starts (it is there: a piece's set holds
// what any state in front of it becomes), a walk over these links in LDS from the chain's seed, then
// the end states and bit offsets of the pieces and the cleared words that k_o1_emit adds to. LDS: 17
// bytes a piece.
__global__ void __launch_bounds__(256) k_o1_sets_walk(O1Chains C, O1Sets B, uint32_t* end_state, uint64_t* bitoff,
                                                      uint64_t* chain_bits, uint32_t* words, uint64_t stride_words,
                                                      uint64_t* failed) {
    extern __shared__ uint8_t link[];
    __shared__ uint64_t part[4];
    __shared__ uint32_t lost;
    const uint32_t q = blockIdx.x, t = threadIdx.x;
    const uint64_t p0 = C.pfirst[q];
    const uint32_t np = (uint32_t)(C.pfirst[q + 1] - p0);
    uint8_t* const pick = link + (uint64_t)np * kSetStates;
    if (t == 0) lost = *failed != 0;  // read once: another chain's workgroup may be setting it
    __syncthreads();
    if (lost) return;
    for (uint32_t u = t; u < np * kSetStates; u += blockDim.x) {
        const uint32_t p = u / kSetStates, k = u % kSetStates;
        uint32_t to = 0xFF;
        if (p + 1 < np && k < B.cnt[p0 + p]) {
            const uint16_t e = B.end[p0 * kSetStates + u];
            const uint32_t m = B.cnt[p0 + p + 1];
            for (uint32_t j = 0; j < m; j++)
                if (B.start[(p0 + p + 1) * kSetStates + j] == e) to = j;
        }
        link[u] = (uint8_t)to;
    }
    __syncthreads();
    if (t == 0) {
        uint32_t cur = 0;
        for (uint32_t p = 0; p < np; p++) {
            pick[p] = (uint8_t)cur;
            cur = link[p * kSetStates + cur];
            if (cur >= kSetStates && p + 1 < np) {
                lost = 1;
                break;
            }
        }
    }
    __syncthreads();
    if (lost) {
        if (t == 0) atomicOr(reinterpret_cast<unsigned long long*>(failed), 1ull);
        return;
    }
    uint64_t base = 0;
    for (uint32_t b = 0; b < np; b += blockDim.x) {
        const uint32_t p = b + t;
        uint64_t bits = 0, sum;
        if (p < np) {
            const uint64_t at = (p0 + p) * kSetStates + pick[p];
            end_state[p0 + p] = B.end[at];
            bits = B.bits[at];
        }
        const uint64_t off = base + block_scan_u64(bits, part, &sum);
        if (p < np) {
            bitoff[p0 + p] = off;
            words[q * stride_words + (off >> 5)] = 0;
        }
        base += sum;
    }
    if (t == 0) {
        chain_bits[q] = base;
        for (uint64_t w = base >> 5; w <= (base + kO1Log + 1) >> 5; w++) words[q * stride_words + w] = 0;
    }
}

// Final state (kO1Log bits) and the end mark of every chain (BIT_closeCStream); byte length out.
__global__ void k_o1_close(const int16_t* bins, O1Chains C, const CTable* ct_all, const uint32_t* end_state,
                           const uint64_t* chain_bits, uint32_t* words, uint64_t stride_words, uint64_t* blen,
                           const uint64_t* failed) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= C.nchains || (failed && *failed)) return;
    const uint64_t lo = C.c[4 * q + 1], hi = C.c[4 * q + 2];
    if (hi <= lo) { blen[q] = 0; return; }
    const CTable* ct = ct_all + C.c[4 * q + 3] * kO1Ctx;
    const uint64_t np = C.pfirst[q + 1] - C.pfirst[q];
    const uint32_t st = np ? end_state[C.pfirst[q + 1] - 1] : o1_seed_state(bins, lo, hi - 1, ct);
    const uint64_t b0 = chain_bits[q];
    WordWriter W{words + q * stride_words, b0 >> 5, 0, (uint32_t)(b0 & 31), true};
    ww_put(W, st, kO1Log);
    ww_put(W, 1, 1);
    if (W.n) { atomicOr(&W.w[W.idx], (uint32_t)W.acc); }
    blen[q] = (b0 + kO1Log + 1 + 7) >> 3;
}


// ---------------------------------------------------------------- method 1 decode
// Decoding tables of every context of every segment, grid (contexts, segments); the counts are read
// from the stream byte by byte (they may sit at any offset). Invalid counts set *err.
__global__ void __launch_bounds__(256) k_o1_dtables(const uint8_t* stream, const uint64_t* nf_off, DEntry* dt_all,
                                                    int* err) {
    __shared__ TableLds L;
    const unsigned t = threadIdx.x;
    const uint8_t* b = stream + nf_off[blockIdx.y] + 2 * ((size_t)blockIdx.x * kO1Sym + t);
    L.norm[t] = (int16_t)(uint16_t)(b[0] | (b[1] << 8));
    __syncthreads();
    DEntry* dt = dt_all + ((size_t)blockIdx.y * kO1Ctx + blockIdx.x) * (1u << kO1Log);
    if (!spread_parallel(L, kO1Log)) {
        if (t == 0) *err = 1;
        // a defined table (state 0, no bits, code 0) so that the decoders stay in range
        for (uint32_t u = t; u < (1u << kO1Log); u += blockDim.x) dt[u] = DEntry{0, 0, 0};
        return;
    }
    // the context that follows each entry's symbol rides in the top four bits of nbBits (15 after an
    // escape, whose context depends on the escaped value); readers mask nbBits with 15
    dtable_parallel(L, kO1Log, dt, [](uint32_t sy) {
        return sy == 255 ? 15u : (uint32_t)o1_ctx((int)((sy >> 1) ^ (~(sy & 1) + 1)));
    });
}


// Exact decoding of a stretch of one chain from a bitstream window staged in LDS, for the walk.
// win[k + kWinPad] holds chain byte wlo + k; the kWinPad bytes below are zero when the window starts at
// the chain's first byte. The decoding tables of contexts hot0 .. hot0 + kWalkCtxN - 1 sit in LDS (hot),
// the others are read from device memory.
constexpr int kWalkCtx0 = 11, kWalkCtxN = 4;  // contexts 11..14: after large codes, where escapes are dense
constexpr int kWinPad = 16;
constexpr int kSeqLanes = 64;       // the sequential decoders run as one wave

struct SeqState {
    int64_t B;      // read position (bits below are unread)
    uint32_t X, cx;
    uint64_t e;     // escapes consumed
    bool bad;
};

// Decodes while the read position stays above `until` (bits), at most `max_n` symbols, for the symbols
// and escapes it counts: escaped codes are read from ov. Returns the symbols decoded.
//
// Per symbol: the table entry (state, context) and the two window words that hold the 32 bits below
// the read position are independent LDS reads; the entry gives the bit count, the next state base,
// the symbol and the next context (top nibble of nbBits; 15 after an escape). Positions are 32-bit
// offsets into the window. One LDS round trip and a few dozen scalar operations per symbol.
__device__ __forceinline__ uint64_t seq_decode(SeqState& S, const FZ_LDS uint8_t* win, int64_t wlo, int64_t until,
                                               uint64_t max_n, const FZ_LDS uint32_t* hot, uint32_t hot0,
                                               const uint32_t* dtg, const int16_t* ov, uint64_t novf) {
    const FZ_LDS uint32_t* w32 = reinterpret_cast<const FZ_LDS uint32_t*>(win);
    const int64_t base = (wlo - kWinPad) * 8;  // bit 0 of the window
    int32_t p = (int32_t)(S.B - base);
    // below 32 bits into the window the word reads would leave it
    const bool raised = until < base + 32;
    const int32_t lim = (int32_t)((raised ? base + 32 : until) - base);
    uint32_t X = S.X, cx = S.cx;
    uint64_t e = S.e;
    const uint32_t kmax = (uint32_t)min<uint64_t>(max_n, 0x7FFFFFFFull);
    uint32_t k = 0;
    while (p > lim && k < kmax) {
        const uint32_t xi = X & ((1u << kO1Log) - 1);
        const uint32_t hc = cx - hot0;
        const int32_t j = (p - 32) >> 5;  // words j, j+1 hold bits [32 j, 32 j + 64), which contain [p - 32, p)
        uint32_t raw = hot[(min(hc, (uint32_t)kWalkCtxN - 1) << kO1Log) + xi];
        const uint64_t w = (uint64_t)w32[j] | ((uint64_t)w32[j + 1] << 32);
        if (hc >= (uint32_t)kWalkCtxN) raw = dtg[((size_t)cx << kO1Log) + xi];
        const uint32_t nb = (raw >> 24) & 15u;
        p -= (int32_t)nb;
        X = (raw & 0xFFFFu) + ((uint32_t)(w >> (uint32_t)(p - 32 * j)) & ((1u << nb) - 1u));
        cx = raw >> 28;
        if (cx == 15u) {
            int code = 32767;
            if (e >= novf) S.bad = true;
            else code = (int)ov[e];
            cx = (uint32_t)o1_ctx(code);
            e++;
        }
        k++;
    }
    // stopped below the staged bytes while symbols remain: the stream runs past its first bit
    if (raised && p <= lim && k < kmax) S.bad = true;
    S.B = base + p;
    S.X = X;
    S.cx = cx;
    S.e = e;
    return k;
}

// Copies chain bytes [w0, hi) into win, where w0 <= lo - kWinPad is the nearest chain byte below
// whose device address is 16-byte aligned, so that whole aligned 16-byte blocks move (one load per
// block; blocks that cross the chain's first or last byte go byte by byte, and bytes outside
// [0, len) read as zero), by one wave. Returns w0: win[i] holds chain byte w0 + i. win must hold
// hi - lo + kWinPad + 32 bytes.
__device__ __forceinline__ int64_t stage_window(FZ_LDS uint8_t* win, const uint8_t* cb, int64_t len, int64_t lo,
                                                int64_t hi) {
    const int64_t s0 = lo - kWinPad;
    const int64_t w0 = s0 - (int64_t)(((uintptr_t)cb + (uintptr_t)s0) & 15u);
    const int64_t nblk = (hi - w0 + 15) / 16;
    // kStageBatch blocks per lane are loaded before any is stored, so their loads are in flight
    // together (a window is a dozen or so blocks per lane)
    constexpr int kStageBatch = 8;
    const int lane = (int)(threadIdx.x & (kSeqLanes - 1));
    for (int64_t q0 = 0; q0 < nblk; q0 += (int64_t)kSeqLanes * kStageBatch) {
        u32x4 v[kStageBatch];
#pragma unroll
        for (int b = 0; b < kStageBatch; b++) {
            const int64_t q = q0 + (int64_t)b * kSeqLanes + lane;
            const int64_t c0 = w0 + 16 * q;
            if (q < nblk && c0 >= 0 && c0 + 16 <= len) {
                v[b] = *reinterpret_cast<const u32x4*>(cb + c0);
            } else if (q < nblk) {
                uint32_t w[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    uint32_t x = 0;
#pragma unroll
                    for (int t = 0; t < 4; t++) {
                        const int64_t i = c0 + 4 * j + t;
                        x |= (i >= 0 && i < len ? (uint32_t)cb[i] : 0u) << (8 * t);
                    }
                    w[j] = x;
                }
                v[b] = u32x4{w[0], w[1], w[2], w[3]};
            } else {
                v[b] = u32x4{0u, 0u, 0u, 0u};
            }
        }
#pragma unroll
        for (int b = 0; b < kStageBatch; b++) {
            const int64_t q = q0 + (int64_t)b * kSeqLanes + lane;
            if (q < nblk) *reinterpret_cast<FZ_LDS u32x4*>(win + 16 * q) = v[b];
        }
    }
    return w0;
}


// ---- order-1 tANS decoding split by bit position ----------------------------------------------
// A chain's bitstream is cut into parts of sub_bits bits. Part r owns the symbols whose decoding
// starts at a read position B in (b_{r+1}, b_r], b_r = pos0 - r * sub_bits; the last one owns
// everything below b_{R-1}. The state in which the true decoder enters a part (its read position is
// 0..12 bits below b_r, tANS state, context) is unknown; what is computed for every part at once is a
// small set of states that holds it:
//  * warm-up (k_o1s_warm): a few decoders per part start at guessed states some thousand symbols ahead
//    of it. Two decoders that meet in position, state and context stay together, so their distinct
//    states at the boundary are few, and the true one is mostly among them.
//  * graphs (k_o1s_graph): every start state of a part is followed to the part's end. The context
//    after an escape depends on the sign of the escaped code, which sits in the side stream at an
//    index that a decoder started mid-chain does not know, so an escape is a node with two out-edges,
//    and decoders that meet at one share it. The states in which the paths leave the part are
//    possible entries of the next one: the following rounds add those that its set lacks. A part
//    whose set holds the true entry so passes it on, and within two or three rounds nearly every set
//    does. Where escapes are frequent the sets saturate after one round: the states that can be
//    reached by any sequence of signs are few tens and contain the true one (512^3 field, REL 1e-3,
//    segment 0, an escape in 48 symbols: 36 states a part at most, 132 nodes on average).
//  * walk (k_o1s_walk, one workgroup per chain): the true path through the graphs with the real escape
//    signs, giving every part its exact entry, escape index and output offset; a part whose set or
//    graph lacks it is decoded exactly on the way.
//  * output (k_o1s_out): every part decodes from its entry into its place.
// States at a part's boundary are packed in 32 bits: bits below the boundary << 17 | context << 13 |
// state; the low 17 bits index the segment's tables.
struct O1Split {
    const uint8_t* cb;    // the chain's bytes
    const uint32_t* dt;   // its segment's tables (DEntry, kO1Ctx x 2^kO1Log)
    const int16_t* ov;    // its escaped codes
    int16_t* out;         // its codes
    int* err;
    uint64_t m, novf;     // codes, escaped codes
    int64_t len, pos0;    // bytes, read position after the initial state
    uint64_t tfirst;      // first part (index over all chains)
    uint64_t cfirst;      // first slot of its candidate arrays (cap a part)
    uint64_t wfirst;      // first warm-up lane (a multiple of 64)
    uint64_t gfirst;      // first graph wave, over all chains
    uint32_t x0, nsub, sub_bits, warm_bits;
    uint32_t lgk;         // 1 << lgk warm-up decoders a part
    uint32_t cap;         // candidates a part holds at most
    uint32_t parts;       // parts a graph wave takes
    uint32_t max_sym;     // symbols an edge may hold
    uint32_t warm_steps;  // pairs of steps a warm-up decoder takes at most
    uint32_t hot0;        // the walk keeps the tables of contexts hot0 .. hot0 + 3 in LDS
    uint32_t cls;         // graph size class
    uint32_t max_nodes;   // nodes a graph wave holds a round
    uint32_t stage;       // nodes of a unit that the walk stages (walk_nodes at most)
};

// Edges: target (16 bits: node, numbered through all rounds of its graph wave, or kSplitExit | exit),
// symbols decoded << 16.
constexpr uint32_t kSplitExit = 0xF000u, kSplitFail = 0xFFFFFFFFu;
constexpr uint32_t kSplitMaxSym = 0xFFFEu;
constexpr int kSplitMaxParts = 16;   // parts a graph wave takes at most
constexpr int kSplitMaxOrig = 256;   // origins it takes at most (parts * cap)

// Arrays shared by the kernels of one decode.
struct O1SplitWs {
    uint32_t* cand;              // start states of every part
    uint32_t* edge;              // their edges
    uint32_t* exits;             // states in which paths leave the part
    uint16_t* hdr;               // [kSplitRounds][parts]: start states | exits << 8 after the round
    uint8_t* n0;                 // [parts]: start states from the warm-up
    uint2* wave;                 // [graph waves][kSplitRounds]: first node in pool (kPoolNone: no room there), nodes
    uint2* pool;                 // nodes: edges for an escaped code >= 0 / < 0
    NodeCount* pool_used;
    uint64_t pool_cap;
    uint64_t nparts;
    uint32_t* res_state;         // [parts]: entry, escape index and output offset on the true path
    uint64_t* res_e;
    uint64_t* res_off;
};

__device__ inline int o1s_chain(const O1Split* ch, int nch, uint64_t x, uint64_t O1Split::*first) {
    int lo = 0, hi = nch;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (ch[mid].*first <= x) lo = mid; else hi = mid;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// Backward bit reader over aligned 32-bit words of a chain: bits [32 j, 32 j + have) are in w (its
// low end first), the word below is in flight. Bits below the chain's first read as zero, as do the
// words below it, which are not touched.
struct ChainWords {
    const uint32_t* d4;   // the aligned word that holds the chain's first byte
    uint32_t m0;          // its bits that belong to the chain
    int32_t shift;        // bit 0 of the chain in it
    __device__ explicit ChainWords(const uint8_t* cb) {
        const uint32_t o = (uint32_t)(uintptr_t)cb & 3u;
        d4 = reinterpret_cast<const uint32_t*>(cb - o);
        m0 = ~0u << (8 * o);
        shift = (int32_t)(8 * o);
    }
    __device__ __forceinline__ uint32_t word(int64_t j) const {
        const uint32_t v = glb(d4)[j < 0 ? 0 : j];
        return j > 0 ? v : (j == 0 ? v & m0 : 0u);
    }
};
struct WordBits {
    uint64_t w;
    int32_t have;
    int64_t j;
    uint32_t nxt;
    // reads from chain bit position B downward (B > 0)
    __device__ __forceinline__ void init(const ChainWords& c, int64_t B) {
        const int64_t a = B + c.shift;
        j = ((a + 31) >> 5) - 2;
        w = ((uint64_t)c.word(j + 1) << 32) | c.word(j);
        have = (int32_t)(a - 32 * j);
        nxt = c.word(j - 1);
    }
    // at least 32 bits; enough for two steps of at most 13
    __device__ __forceinline__ void refill(const ChainWords& c) {
        if (have < 32) {
            w = (w << 32) | nxt;
            have += 32;
            j--;
            nxt = c.word(j - 1);
        }
    }
    __device__ __forceinline__ uint32_t take(uint32_t nb) {
        have -= (int32_t)nb;
        return (uint32_t)(w >> ((uint32_t)have & 63u)) & ((1u << nb) - 1u);
    }
};

// Guessed start states: any spread will do, the same ones in every run.
__device__ __forceinline__ uint32_t o1s_mix(uint32_t x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    return x ^ (x >> 16);
}

// One lane per guessed decoder; the 2^lgk lanes of a part sit in one wave and drop duplicates at the
// boundary. After an escape each lane picks a sign at random, so that lanes which have met can part
// again and cover the states reachable by other signs.
__global__ void __launch_bounds__(256) k_o1s_warm(const O1Split* ch, int nch, uint64_t nlanes, O1SplitWs ws) {
    const uint64_t g = (uint64_t)xcd_block() * blockDim.x + threadIdx.x;
    if (g >= nlanes) return;  // whole waves: nlanes is a multiple of 64
    const O1Split& c = ch[o1s_chain(ch, nch, g & ~63ull, &O1Split::wfirst)];
    const uint32_t K = 1u << c.lgk;
    const uint64_t local = g - c.wfirst;
    const uint64_t r = local >> c.lgk;
    const uint32_t k = (uint32_t)local & (K - 1);
    const bool valid = r > 0 && r < c.nsub;
    uint32_t state = ~0u;
    if (valid) {
        const ChainWords cw(c.cb);
        const uint32_t* dt = c.dt;
        const int64_t b = c.pos0 - (int64_t)r * c.sub_bits;
        uint32_t seed = o1s_mix((uint32_t)local * 2654435761u + 12345u);
        int64_t B = b + c.warm_bits;
        uint32_t idx;
        if (B >= c.pos0) {  // near the chain's start: from its true state
            B = c.pos0;
            idx = c.x0 & ((1u << kO1Log) - 1);
        } else {
            B -= seed % 13u;
            idx = (((seed >> 8) % (uint32_t)kO1Ctx) << kO1Log) | ((seed >> 16) & ((1u << kO1Log) - 1));
        }
        int32_t rem = (int32_t)(B - b);
        WordBits rd;
        rd.init(cw, B);
        // a context whose one symbol reads no bits would never get there
        uint32_t guard = c.warm_steps;
        auto step = [&]() {
            if (rem <= 0) return;
            const uint32_t raw = glb(dt)[idx];
            const uint32_t nb = (raw >> 24) & 15u;
            rem -= (int32_t)nb;
            const uint32_t x = (raw & ((1u << kO1Log) - 1)) + rd.take(nb);
            uint32_t cx = raw >> 28;
            if (cx == 15u) {
                seed = seed * 1664525u + 1013904223u;
                cx = 13u + (seed >> 31);
            }
            idx = (cx << kO1Log) | (x & ((1u << kO1Log) - 1));
        };
        while (rem > 0 && guard--) {
            rd.refill(cw);
            step();
            step();
        }
        if (rem <= 0) state = ((uint32_t)-rem << 17) | idx;
    }
    bool keep = state != ~0u;
    const int lane = threadIdx.x & 63, base = lane & ~(int)(K - 1);
    for (uint32_t i = 0; i < K; i++) {
        const uint32_t o = __shfl(state, base + (int)i);
        keep = keep && !(i < k && o == state);
    }
    const uint64_t grp = (K == 64 ? ~0ull : ((1ull << K) - 1) << base) & __ballot(keep);
    const uint32_t n = min((uint32_t)__popcll(grp), c.cap);
    const uint32_t at = (uint32_t)__popcll(grp & ((1ull << lane) - 1));
    const uint64_t slot = c.cfirst + r * c.cap;
    if (r == 0 && k == 0) {
        ws.cand[slot] = c.x0 & ((1u << kO1Log) - 1);  // the chain starts in context 0
        ws.n0[c.tfirst] = 1;
    }
    if (valid) {
        if (keep && at < c.cap) ws.cand[slot + at] = state;
        if (k == 0) ws.n0[c.tfirst + r] = (uint8_t)n;
    }
}

// The graphs of the parts of one wave, from this round's new start states. A lane takes one edge at a
// time (a start state, or a node and a sign), decodes to the next escape or the part's end, and looks
// the state it met up in a hash table in LDS: a new escape state is a new node and two more edges. The
// edges still to take are the tail of the node list, so there is no queue. Parts share a wave where
// their edges are few (chains without escapes have a handful of start states). Steps run eight at a
// time between looks at the table; a lane that has met its end waits for the rest.
// NC: nodes a wave holds at most (c.max_nodes is no more); past it, and where a table or the pool is full, the edges left stay
// marked and the walk decodes such parts exactly.
template <int NC>
__global__ void __launch_bounds__(64) k_o1s_graph(const O1Split* ch, int nch, uint32_t nwaves, int round, O1SplitWs ws) {
    constexpr uint32_t kSlots = NC <= 128 ? 512 : 2 * NC;
    __shared__ unsigned long long key[kSlots];  // 1 << 63 | part << 43 | (bits above the end + 64) << 17 | ctx << 13 | state
    __shared__ uint16_t val[kSlots];            // node, or kSplitExit | exit
    __shared__ uint16_t list[NC];               // node -> slot
    __shared__ uint2 nodes[NC];
    __shared__ uint32_t ost[kSplitMaxOrig];
    __shared__ uint16_t oat[kSplitMaxOrig];     // part << 8 | slot
    __shared__ uint32_t nex[kSplitMaxParts], ncand[kSplitMaxParts];
    const uint32_t l = threadIdx.x;
    const uint64_t below = (1ull << l) - 1;
    if (xcd_block() >= nwaves) return;
    const uint64_t gw = ch[0].gfirst + xcd_block();
    const O1Split& c = ch[o1s_chain(ch, nch, gw, &O1Split::gfirst)];
    const uint32_t wl = (uint32_t)(gw - c.gfirst);
    const uint32_t p0 = wl * c.parts;
    const uint32_t np = min(c.parts, c.nsub - 1 - p0);  // the last part has no graph
    const uint32_t cap = c.cap;
    const uint64_t t0 = c.tfirst + p0, c0 = c.cfirst + (uint64_t)p0 * cap;
    uint16_t* hdr = ws.hdr + (uint64_t)round * ws.nparts;
    for (uint32_t i = l; i < kSlots; i += 64) key[i] = 0;
    // this round's start states
    uint32_t no = 0;
    for (uint32_t p = 0; p < np; p++) {
        const uint64_t t = t0 + p, cs = c0 + (uint64_t)p * cap;
        uint32_t n = 0, ne = 0;
        if (round == 0) {
            n = ws.n0[t];
            for (uint32_t i = l; i < n; i += 64) {
                ost[no + i] = ws.cand[cs + i];
                oat[no + i] = (uint16_t)(p << 8 | i);
            }
            no += n;
        } else {
            const uint32_t h = (hdr - ws.nparts)[t];
            n = h & 255u;
            ne = h >> 8;
            if (p0 + p > 0) {
                // exits of the part before that its latest round added, less those already in the set
                const uint32_t e1 = (hdr - ws.nparts)[t - 1] >> 8;
                const uint32_t e0 = round > 1 ? (hdr - 2 * ws.nparts)[t - 1] >> 8 : 0u;
                const uint32_t nold = n;
                for (uint32_t i0 = e0; i0 < e1; i0 += 64) {
                    const uint32_t i = i0 + l;
                    bool keep = i < e1;
                    const uint32_t x = keep ? ws.exits[cs - cap + i] : 0u;
                    for (uint32_t q = 0; q < nold; q++) keep = keep && ws.cand[cs + q] != x;
                    const uint64_t mk = __ballot(keep);
                    const uint32_t at = n + (uint32_t)__popcll(mk & below);
                    if (keep && at < cap) {
                        ws.cand[cs + at] = x;
                        ost[no + (at - n)] = x;
                        oat[no + (at - n)] = (uint16_t)(p << 8 | at);
                    }
                    const uint32_t add = min((uint32_t)__popcll(mk), cap - n);
                    n += add;
                    no += add;
                }
            }
        }
        if (l == 0) {
            ncand[p] = n;
            nex[p] = ne;
        }
    }
    __syncthreads();
    uint32_t id0 = 0;  // nodes of earlier rounds
    for (int z = 0; z < round; z++) id0 += ws.wave[gw * kSplitRounds + z].y;
    if (no == 0) {
        for (uint32_t p = l; p < np; p += 64) hdr[t0 + p] = (uint16_t)(ncand[p] | nex[p] << 8);
        if (l == 0) ws.wave[gw * kSplitRounds + round] = make_uint2(0, 0);
        return;
    }
    for (uint32_t i = l; i < no; i += 64) ws.edge[c0 + (uint64_t)(oat[i] >> 8) * cap + (oat[i] & 255u)] = kSplitFail;
    // returns the slot of k, and whether it was put there now; kSlots: the table is full
    auto insert = [&](unsigned long long k, bool& fresh) -> uint32_t {
        uint32_t s = ((uint32_t)(k >> 32) * 0x9E3779B1u ^ (uint32_t)k * 0x85EBCA6Bu) >> 8;
        fresh = false;
        for (int q = 0; q < 128; q++, s++) {
            s &= kSlots - 1;
            const unsigned long long old = atomicCAS(&key[s], 0ull, k);
            if (old == 0) { fresh = true; return s; }
            if (old == k) return s;
        }
        return kSlots;
    };
    // exits of earlier rounds
    if (round > 0)
        for (uint32_t p = 0; p < np; p++)
            for (uint32_t i = l; i < nex[p]; i += 64) {
                const uint32_t x = ws.exits[c0 + (uint64_t)p * cap + i];
                bool fresh;
                const uint32_t s = insert(1ull << 63 | (unsigned long long)p << 43 |
                                              (unsigned long long)(64u - (x >> 17)) << 17 | (x & 0x1FFFFu), fresh);
                if (s < kSlots) val[s] = (uint16_t)(kSplitExit | i);
            }
    __syncthreads();
    const ChainWords cw(c.cb);
    const uint32_t* dt = c.dt;
    const int64_t stop0 = c.pos0 - (int64_t)(p0 + 1) * c.sub_bits;  // end of the wave's first part
    uint32_t head = 0, tail = no, nn = 0;  // edges taken, edges known, nodes
    bool active = false;
    uint32_t task = 0, p = 0, idx = 0, nsym = 0;
    int32_t rem = 0;
    WordBits rd{0, 0, 0, 0};
    for (;;) {
        const uint64_t idle = __ballot(!active);
        const uint32_t mine = head + (uint32_t)__popcll(idle & below);
        bool run = active;
        if (!active && mine < tail) {
            task = mine;
            if (task < no) {
                const uint32_t x = ost[task];
                p = oat[task] >> 8;
                rem = (int32_t)c.sub_bits - (int32_t)(x >> 17);
                idx = x & 0x1FFFFu;
            } else {
                const uint32_t q = task - no;
                const unsigned long long k = key[list[q >> 1]];
                p = (uint32_t)(k >> 43) & 15u;
                rem = (int32_t)((uint32_t)(k >> 17) & 0x3FFFFFFu) - 64;
                idx = ((13u + (q & 1u)) << kO1Log) | ((uint32_t)k & ((1u << kO1Log) - 1));
            }
            nsym = 0;
            active = true;
            run = rem > 0;
            if (run) rd.init(cw, stop0 - (int64_t)p * c.sub_bits + rem);
        }
        head = min(tail, head + (uint32_t)__popcll(idle));
        if (__ballot(active) == 0) break;
        bool esc = false, dead = false;
        auto step = [&]() {
            if (!run) return;
            const uint32_t raw = glb(dt)[idx];
            const uint32_t nb = (raw >> 24) & 15u;
            rem -= (int32_t)nb;
            const uint32_t x = (raw + rd.take(nb)) & ((1u << kO1Log) - 1);
            idx = (raw >> 28 << kO1Log) | x;
            nsym++;
            esc = raw >> 28 == 15u;
            run = rem > 0 && !esc;
        };
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (run) rd.refill(cw);
            step();
            step();
        }
        if (run && nsym > c.max_sym) {
            run = false;
            dead = true;  // a stretch of many symbols in few bits: the walk takes it
        }
        // lanes that met an escape or the end
        const bool ev = active && !run;
        if (__ballot(ev) == 0) continue;
        bool fresh = false;
        uint32_t slot = kSlots;
        if (ev && !dead)
            slot = insert(1ull << 63 | (unsigned long long)p << 43 | (unsigned long long)(uint32_t)(rem + 64) << 17 |
                              (idx | (esc ? 0xFu << kO1Log : 0u)), fresh);
        const uint64_t nmask = __ballot(fresh && esc);
        const uint32_t id = nn + (uint32_t)__popcll(nmask & below);
        const bool full = nn + (uint32_t)__popcll(nmask) > c.max_nodes;
        if (fresh) {
            if (esc) {
                if (id < (uint32_t)NC) {
                    val[slot] = (uint16_t)(id0 + id);
                    list[id] = (uint16_t)slot;
                    nodes[id] = make_uint2(kSplitFail, kSplitFail);
                }
            } else {
                const uint32_t e = atomicAdd(&nex[p], 1u);
                if (e < cap) {
                    ws.exits[c0 + (uint64_t)p * cap + e] = ((uint32_t)-rem << 17) | idx;
                    val[slot] = (uint16_t)(kSplitExit | e);
                } else {
                    val[slot] = 0xFFFFu;
                }
            }
        }
        __syncthreads();
        if (full) break;
        if (ev) {
            const uint32_t v = slot < kSlots ? val[slot] : 0xFFFFu;
            const uint32_t e = v == 0xFFFFu || nsym > kSplitMaxSym ? kSplitFail : v | nsym << 16;
            if (task < no) ws.edge[c0 + (uint64_t)(oat[task] >> 8) * cap + (oat[task] & 255u)] = e;
            else if ((task - no) & 1u) nodes[(task - no) >> 1].y = e;
            else nodes[(task - no) >> 1].x = e;
            active = false;
        }
        nn += (uint32_t)__popcll(nmask);
        tail = no + 2 * nn;
        __syncthreads();
    }
    __syncthreads();
    nn = min(nn, (uint32_t)NC);
    uint32_t at = 0;
    if (nn) {
        if (l == 0) at = pool_first(atomicAdd(ws.pool_used, (NodeCount)nn), nn, ws.pool_cap);
        at = __builtin_amdgcn_readfirstlane(at);
        if (at != kPoolNone)  // else the walk finds no node and decodes such parts exactly
            for (uint32_t i = l; i < nn; i += 64) ws.pool[at + i] = nodes[i];
    }
    if (l == 0) ws.wave[gw * kSplitRounds + round] = make_uint2(at, nn);
    for (uint32_t i = l; i < np; i += 64) hdr[t0 + i] = (uint16_t)(ncand[i] | min(nex[i], cap) << 8);
}

// One workgroup per chain; wave 0 walks, the others stage what it needs next in LDS: the sets and nodes
// of whole graph waves ("units" of c.parts parts), a buffer of units while the walk is in the other.
// The walk is one LDS round trip per escape and three per part. A part that the graph does not hold is
// decoded exactly; the tables of four contexts then take the place of both buffers. (Staging one part at
// a time, behind two dependent device loads, cost 1.5 us a part and 0.35 us an escape: 512^3 field at
// REL 1e-3 23.2 ms a call, counts of 101 x 128 x 150 11.3 ms.)
constexpr int kWalkThreads = 512;
constexpr uint32_t kWalkBuf = 65536;   // bytes of one buffer
constexpr int64_t kWalkStage = 4096;   // bitstream bytes staged per window of an exact decode
// Nodes of a unit that are staged at most, by size class; the rest are read from memory.
__host__ __device__ constexpr uint32_t walk_nodes(uint32_t cls) { return cls == 0 ? 64u : cls == 1 ? 512u : 1024u; }

__global__ void __launch_bounds__(kWalkThreads) k_o1s_walk(const O1Split* ch, int nch, O1SplitWs ws, unsigned int* stats) {
    __shared__ __align__(16) uint32_t mem[2 * kWalkBuf / 4];  // two buffers, or the hot tables
    __shared__ __align__(16) uint32_t stage32[(kWalkStage + kWinPad + 32) / 4 + 4];
    __shared__ uint32_t sh_miss, sh_stop;
    static_assert(2 * kWalkBuf / 4 >= (uint32_t)kWalkCtxN << kO1Log, "the tables fit in the buffers");
    const int q = blockIdx.x;
    if (q >= nch) return;
    const O1Split c = ch[q];
    const uint32_t tid = threadIdx.x, l = tid & 63u, wv = tid >> 6;
    const bool lead = tid == 0;
    const uint32_t P = c.parts, pc = P * c.cap;  // candidates of a unit
    const uint32_t NS = walk_nodes(c.cls);  // (a number from c, read in its place, makes the hops 2.5% slower)
    // a unit's words: nodes (first, for their alignment), cand, edge, exits, start states of each part,
    // nodes staged
    const uint32_t o_cand = 2 * NS, o_edge = o_cand + pc, o_exit = o_edge + pc, o_n = o_exit + pc,
                   o_ns = o_n + kSplitMaxParts, unit_words = o_ns + 4;
    const uint32_t U = (kWalkBuf / 4) / unit_words;  // units a buffer
    const uint32_t ngraph = c.nsub - 1, nunit = (ngraph + P - 1) / P;
    const uint16_t* hdr = ws.hdr + (uint64_t)(kSplitRounds - 1) * ws.nparts + c.tfirst;
    FZ_LDS uint32_t* const lmem = lds(mem);
    const FZ_GLB u32x2* pool = glb(reinterpret_cast<const u32x2*>(ws.pool));
    auto stage_units = [&](uint32_t u0, FZ_LDS uint32_t* buf, uint32_t w0, uint32_t nw) {  // by waves w0 .. w0 + nw - 1
        const uint32_t u1 = min(nunit, u0 + U);
        for (uint32_t u = u0 + (wv - w0); u < u1; u += nw) {
            FZ_LDS uint32_t* b = buf + (u - u0) * unit_words;
            const uint2* rw = ws.wave + (c.gfirst + u) * kSplitRounds;
            uint2 rd[kSplitRounds];
#pragma unroll
            for (int z = 0; z < kSplitRounds; z++) rd[z] = rw[z];
            // the last unit's sets end with the chain's
            const uint64_t cs = c.cfirst + (uint64_t)u * pc;
            const uint32_t nc = min(pc, (c.nsub - u * P) * c.cap);
            for (uint32_t i = l; i < nc; i += 128) {
                const uint32_t k = min(i + 64, nc - 1);
                const uint32_t v0 = glb(ws.cand)[cs + i], v1 = glb(ws.edge)[cs + i], v2 = glb(ws.exits)[cs + i];
                const uint32_t v3 = glb(ws.cand)[cs + k], v4 = glb(ws.edge)[cs + k], v5 = glb(ws.exits)[cs + k];
                b[o_cand + i] = v0;
                b[o_edge + i] = v1;
                b[o_exit + i] = v2;
                b[o_cand + k] = v3;
                b[o_edge + k] = v4;
                b[o_exit + k] = v5;
            }
            if (l < P && u * P + l < ngraph) b[o_n + l] = glb(hdr)[u * P + l] & 255u;
            // the nodes of all rounds, one after another, eight loads a lane in flight
            uint32_t ns = 0;
            bool room = true;
#pragma unroll
            for (int z = 0; z < kSplitRounds; z++) {
                const uint32_t n = room && rd[z].x != kPoolNone ? min(rd[z].y, c.stage - ns) : 0u;
                for (uint32_t i0 = 0; i0 < n; i0 += 512) {
                    u32x2 v[8];
#pragma unroll
                    for (int j = 0; j < 8; j++) v[j] = pool[rd[z].x + min(i0 + 64u * j + l, n - 1)];
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        if (i0 + 64u * j + l < n) {
                            b[2 * (ns + i0 + 64u * j + l)] = v[j].x;
                            b[2 * (ns + i0 + 64u * j + l) + 1] = v[j].y;
                        }
                }
                room = room && n == rd[z].y;
                ns += n;
            }
            if (l == 0) b[o_ns] = ns;
        }
    };
    // an edge of a node that is not staged
    auto far_edge = [&](uint32_t u, uint32_t tgt, uint32_t neg) -> uint32_t {
        const uint2* rw = ws.wave + (c.gfirst + u) * kSplitRounds;
        for (int z = 0; z < kSplitRounds; z++) {
            const uint2 v = rw[z];
            if (tgt < v.y) return v.x == kPoolNone ? kSplitFail : glb(reinterpret_cast<const uint32_t*>(ws.pool))[2 * ((uint64_t)v.x + tgt) + neg];
            tgt -= v.y;
        }
        return kSplitFail;
    };
    uint32_t cur = c.x0 & ((1u << kO1Log) - 1);
    uint64_t e = 0, off = 0;
    // signs of 64 escaped codes from index eb on (bit k: code eb + k is negative), the next 64 in flight
    uint64_t eb = 0, signs = 0;
    int vnext = 0;
    auto sign_load = [&](uint64_t at) { return at + l < c.novf ? (int)glb(c.ov)[at + l] : 0; };
    if (wv == 0) {
        signs = __ballot(sign_load(0) < 0);
        vnext = sign_load(64);
    }
    uint32_t r = 0;        // part the walk is at
    uint32_t u0 = 0, cb = 0;  // first unit of the current buffer, which one it is
    const uint32_t nwaves = kWalkThreads / 64;
    if (ngraph) stage_units(0, lmem, 0, nwaves);
    if (lead) sh_stop = 0;
    while (r < ngraph) {
        if (lead) sh_miss = 0;
        __syncthreads();
        const uint32_t r_end = min(ngraph, (u0 + U) * P);
        if (wv > 0) {
            stage_units(u0 + U, lmem + (cb ^ 1u) * (kWalkBuf / 4), 1, nwaves - 1);
        } else {
            const FZ_LDS uint32_t* buf = lmem + cb * (kWalkBuf / 4);
            uint32_t u = u0, pu = r - u0 * P;
            while (pu >= P) { pu -= P; u++; }
            bool miss = false;
            for (; r < r_end; r++) {
                const FZ_LDS uint32_t* b = buf + (u - u0) * unit_words;
                if (lead) {
                    ws.res_state[c.tfirst + r] = cur;
                    ws.res_e[c.tfirst + r] = e;
                    ws.res_off[c.tfirst + r] = off;
                }
                const uint32_t n = __builtin_amdgcn_readfirstlane(b[o_n + pu]);
                const uint32_t ns = __builtin_amdgcn_readfirstlane(b[o_ns]);
                uint32_t ed = kSplitFail;
                bool found = false;
                for (uint32_t i = 0; i < n && !found; i += 64) {
                    const uint64_t mk = __ballot(i + l < n && b[o_cand + pu * c.cap + i + l] == cur);
                    if (mk) {
                        found = true;
                        ed = b[o_edge + pu * c.cap + i + (uint32_t)__builtin_ctzll(mk)];
                    }
                }
                ed = __builtin_amdgcn_readfirstlane(ed);
                // every escape is one hop: node, sign, next edge. All of it is wave-uniform and kept in
                // scalar registers; signs holds those of 64 escapes, k the next one's place in it
                uint64_t pe = uniform64(e), sg = uniform64(signs);
                uint64_t po = off + (ed >> 16);
                uint32_t tgt = ed & 0xFFFFu, k = uniform32((uint32_t)min<uint64_t>(pe - eb, 128)), guard = 0;
                while (tgt < kSplitExit) {
                    if (k >= 64) {
                        if (k < 128) {
                            eb += 64;
                            k -= 64;
                            signs = __ballot(vnext < 0);
                        } else {
                            eb = pe;
                            k = 0;
                            signs = __ballot(sign_load(eb) < 0);
                        }
                        vnext = sign_load(eb + 64);
                        sg = uniform64(signs);
                    }
                    const uint32_t k0 = k;
                    uint32_t sum = 0;
                    if (tgt < ns) {
                        do {
                            ed = uniform32(b[2 * tgt + ((uint32_t)(sg >> k) & 1u)]);
                            sum += ed >> 16;
                            tgt = ed & 0xFFFFu;
                            k++;
                        } while (tgt < ns && k < 64);
                    } else {
                        ed = uniform32(far_edge(u, tgt, (uint32_t)(sg >> k) & 1u));
                        sum = ed >> 16;
                        tgt = ed & 0xFFFFu;
                        k++;
                    }
                    po += sum;
                    pe += k - k0;
                    guard += k - k0;
                    if (guard > 65536u) {  // a loop of escapes that read no bits
                        ed = kSplitFail;
                        break;
                    }
                }
                if (ed == kSplitFail) {
                    if (lead) {
                        atomicAdd(&stats[found ? 0 : 1], 1u);  // no whole path in the graph / entry not in the set
                        atomicAdd(&stats[6 + q], 1u);          // per chain
                    }
                    miss = true;
                    break;
                }
                cur = __builtin_amdgcn_readfirstlane(b[o_exit + pu * c.cap + (ed & 0xFFFu)]);
                e = pe;
                off = po;
                if (off > c.m) {  // a corrupt stream
                    if (lead) {
                        *c.err = 1;
                        sh_stop = 1;
                    }
                    break;
                }
                if (++pu == P) { pu = 0; u++; }
            }
            if (lead) sh_miss = miss ? r + 1 : 0;
        }
        __syncthreads();
        if (sh_stop) return;
        const uint32_t miss = sh_miss;
        if (!miss) {
            u0 += U;
            cb ^= 1u;
            r = r_end;
            continue;
        }
        // exact decode of part r = miss - 1, the bitstream staged in LDS window by window
        r = miss - 1;
        for (uint32_t i = tid; i < (uint32_t)kWalkCtxN << kO1Log; i += kWalkThreads)
            mem[i] = glb(c.dt)[((size_t)c.hot0 << kO1Log) + i];
        __syncthreads();
        if (wv == 0) {
            const int64_t b = c.pos0 - (int64_t)r * c.sub_bits, stop = b - c.sub_bits;
            SeqState z{b - (int64_t)(cur >> 17), cur & ((1u << kO1Log) - 1), (cur >> kO1Log) & 15u, e, false};
            uint8_t* st8 = reinterpret_cast<uint8_t*>(stage32);
            while (z.B > stop && off < c.m && !z.bad) {
                const int64_t hi = min<int64_t>(c.len, (z.B + 7) / 8 + 1);
                const int64_t lo = max<int64_t>(0, hi - kWalkStage);
                wave_lds_order();
                const int64_t w0 = stage_window(lds(st8), c.cb, c.len, lo, hi);
                wave_lds_order();
                // window reads reach 64 bits below the read position: stay above the staged bytes
                // unless they start at the chain's first byte
                const int64_t floor_bits = lo == 0 ? INT64_MIN : lo * 8 + 64;
                off += seq_decode(z, lds(st8), w0 + kWinPad, max<int64_t>(stop, floor_bits), c.m - off, lds(mem), c.hot0,
                                  c.dt, c.ov, c.novf);
            }
            e = z.e;
            const int64_t d = stop - z.B;
            if (z.bad || d < 0 || d > 12 || off > c.m) {  // a corrupt stream: its codes ran out inside the part
                if (lead) {
                    *c.err = 1;
                    sh_stop = 1;
                }
            }
            cur = ((uint32_t)d & 15u) << 17 | z.cx << kO1Log | (z.X & ((1u << kO1Log) - 1));
        }
        __syncthreads();
        if (sh_stop) return;
        r++;
        u0 = r / P;
        cb = 0;
        if (r < ngraph) stage_units(u0, lmem, 0, nwaves);
    }
    if (lead) {  // the last part
        ws.res_state[c.tfirst + r] = cur;
        ws.res_e[c.tfirst + r] = e;
        ws.res_off[c.tfirst + r] = off;
    }
}

// Final pass: every part decodes from its entry into its place in the code array. Its code count is
// the distance to the next part's output offset, so codes leave in aligned 64-byte runs (32 codes
// packed in registers, four 16-byte stores) between a head and a tail written one by one.
__global__ void __launch_bounds__(256) k_o1s_out(const O1Split* ch, int nch, O1SplitWs ws) {
    const uint64_t t = (uint64_t)xcd_block() * blockDim.x + threadIdx.x;
    if (t >= ws.nparts) return;
    int q = 0;
    {
        int hi = nch;
        while (hi - q > 1) {
            const int mid = (q + hi) >> 1;
            if (ch[mid].tfirst <= t) q = mid; else hi = mid;
        }
    }
    const O1Split& c = ch[q];
    if (*c.err) return;  // the walk stopped short: entries are missing
    const uint64_t r = t - c.tfirst;
    const bool last = r + 1 >= c.nsub;
    const uint64_t m = c.m;
    const uint64_t o0 = ws.res_off[t], o1 = last ? m : ws.res_off[t + 1];
    if (o0 > o1 || o1 > m) {  // offsets from a corrupt stream
        *c.err = 1;
        return;
    }
    const uint32_t s = ws.res_state[t];
    uint64_t e = ws.res_e[t];
    const uint64_t novf = c.novf;
    const uint32_t* dt = c.dt;
    const int16_t* ov = c.ov;
    const ChainWords cw(c.cb);
    const int64_t b = c.pos0 - (int64_t)r * c.sub_bits, B0 = b - (int64_t)(s >> 17);
    uint32_t idx = s & 0x1FFFFu;
    WordBits rd;
    rd.init(cw, B0);
    bool bad = false;
    uint32_t nb = 0;  // bits of the latest symbol
    auto step = [&]() -> uint32_t {
        const uint32_t raw = glb(dt)[idx];
        nb = (raw >> 24) & 15u;
        const uint32_t x = (raw + rd.take(nb)) & ((1u << kO1Log) - 1);
        uint32_t cx = raw >> 28;
        const uint32_t sy = (raw >> 16) & 0xFFu;
        int code = (int)((sy >> 1) ^ (~(sy & 1) + 1));
        if (cx == 15u) {
            if (e < novf) code = glb(ov)[e];
            else { code = 32767; bad = true; }
            e++;
            cx = (uint32_t)o1_ctx(code);
        }
        idx = (cx << kO1Log) | x;
        return (uint32_t)code & 0xFFFFu;
    };
    int16_t* out = c.out;
    uint64_t i = o0;
    const uint64_t iend = o1;
    const uint64_t a0 = ((uintptr_t)out >> 1) & 31;  // 64-byte alignment of the code array
    while (i < iend && ((i + a0) & 31)) {
        rd.refill(cw);
        out[i++] = (int16_t)step();
    }
    while (i + 32 <= iend) {
        uint32_t w[16];
#pragma unroll
        for (int j = 0; j < 16; j++) {
            rd.refill(cw);
            const uint32_t a = step();
            w[j] = a | (step() << 16);
        }
        uint32_t* o = reinterpret_cast<uint32_t*>(out + i);
#pragma unroll
        for (int j = 0; j < 16; j += 4)
            *reinterpret_cast<u32x4*>(o + j) = u32x4{w[j], w[j + 1], w[j + 2], w[j + 3]};
        i += 32;
    }
    while (i < iend) {
        rd.refill(cw);
        out[i++] = (int16_t)step();
    }
    // the part's symbols are those that start above the next boundary, and leave the state and the
    // escape that the walk entered the next part with
    const int64_t pos = 32 * rd.j + rd.have - cw.shift, stop = b - (int64_t)c.sub_bits;
    if (last) {
        bad = bad || e != novf;
    } else {
        const uint32_t to = ws.res_state[t + 1];
        bad = bad || pos != stop - (int64_t)(to >> 17) || idx != (to & 0x1FFFFu) || e != ws.res_e[t + 1] ||
              (o1 > o0 && pos + (int64_t)nb <= stop);
    }
    if (bad) *c.err = 1;
}

// ---- chains decoded from their start ------------------------------------------------------------
// Chains that cannot be split (dense escapes, or few bits a symbol) are decoded by one workgroup each,
// from the first symbol to the last. What bounds them is one dependent table lookup after another, so
// the wave that makes the lookups (wave 0) does nothing else: it logs the states it goes through, and
// of the other waves one turns a log into codes (symbols, escaped values, places in the output) while
// the next is being written, and one stages bits and escape signs ahead.
//
// Lookups go to re-encoded tables, four contexts of them in LDS, the others in device memory. Entry:
//   [4:0]   31 - bits read: the shift that brings them down from the top of the 31 next bits
//   [8:5]   bits read
//   [12:9]  context after the symbol where it is not in LDS (15: an escape)
//   [13]    an escape, with both contexts that can follow in slots 0 and 1: the sign of the escaped
//           value, held at the same bit, picks one
//   [14]    the next lookup is not in LDS (or an escape whose contexts are not in slots 0 and 1)
//   [31:16] slot << 13 | next state less the bits read
// so the next address is three operations from the entry, and everything else (bit buffer, sign
// register, test for the rare path) fits under the latency of the LDS read. Measured on the 512^3 field
// at REL 1e-4, 60 chains of 2.24 M symbols with an escape in two, 3% of the lookups not in LDS: 134 ms
// (60 ns a symbol; 204 ms with one wave for all of it).
// Symbols of more than half probability read no bits most of the time. In chains of few bits a symbol
// an entry stands for up to kSerialRun such steps and the one after them (they need no bits, so the
// state alone decides them): the log then holds one state for all of them, and its expansion walks
// them again, 64 states at a time. Measured on the 256x384x384 float64 front field (0.3-0.4 bits a
// symbol, 4 to 5 symbols a lookup): 39 ms (202 ms).
constexpr uint32_t kSerialSlow = 1u << 14, kSerialEsc = 1u << 13;
constexpr int kSerialHot = 4;            // contexts in LDS
constexpr int kSerialRun = 7;            // steps without bits an entry stands for at most
constexpr uint32_t kSerialGroup = 6;     // steps between refills of the bit buffer
constexpr uint32_t kSerialLog = 1020;    // states a round logs at most
constexpr uint32_t kSerialRing = 2048;   // words of bitstream in LDS: two rounds of 13 bits a step and more
constexpr uint32_t kSerialSigns = 128;   // words of escape signs in LDS, likewise
constexpr int kSerialThreads = 192;
// Log values: the byte address of a state's entry in LDS, or one of these and (context << 13 | state) << 2
// for an entry in device memory or a single step.
constexpr uint32_t kLogCold = 1u << 22, kLogSingle = 1u << 23;

// Which contexts of a segment are in LDS: perm(slot) for slots 0 .. 3, inv(context) its slot (4 and more:
// not there). esc: contexts 13 and 14 are in slots 0 and 1.
struct SerialMap {
    uint64_t inv_nibbles;
    uint32_t perm_bytes;
    uint32_t esc;
    uint32_t run;  // steps without bits an entry takes in
    uint32_t pad;
    __host__ __device__ uint32_t inv(uint32_t c) const { return (uint32_t)(inv_nibbles >> (4 * c)) & 15u; }
    __host__ __device__ uint32_t perm(uint32_t slot) const { return (perm_bytes >> (8 * slot)) & 255u; }
};
struct SerialTables {   // one segment's tables to re-encode
    const uint32_t* dt;
    uint32_t* et;
    SerialMap map;
};
struct SerialJob {
    const uint8_t* cb;   // the chain's bytes
    const uint32_t* dt;  // its segment's decoding tables
    const uint32_t* et;  // the re-encoded ones, by context
    const int16_t* ov;   // its escaped codes
    int16_t* out;        // its codes
    int* err;
    uint64_t* times;     // statistics: 100 MHz clock at its start and end (or null)
    uint64_t m, novf;    // codes, escaped codes
    int64_t pos0;        // read position after the initial state
    uint32_t x0;         // initial state
    uint32_t pad;
    SerialMap map;
};

// grid (contexts, segments)
__global__ void __launch_bounds__(256) k_o1d_tables(const SerialTables* tabs) {
    const SerialTables& t = tabs[blockIdx.y];
    const SerialMap dm = t.map;
    const FZ_GLB uint32_t* dt = glb(t.dt);
    for (uint32_t i = threadIdx.x; i < (1u << kO1Log); i += blockDim.x) {
        uint32_t raw = dt[blockIdx.x << kO1Log | i];
        for (uint32_t k = 0; k < dm.run && (raw >> 24) < 0xF0u && ((raw >> 24) & 15u) == 0; k++)
            raw = dt[raw >> 28 << kO1Log | (raw & ((1u << kO1Log) - 1))];
        const uint32_t nb = (raw >> 24) & 15u, ns = raw & ((1u << kO1Log) - 1), cx = raw >> 28;
        uint32_t e = (31u - nb) | nb << 5 | ns << 16;
        if (cx == 15u) e |= dm.esc ? kSerialEsc : kSerialSlow | 15u << 9;
        else if (dm.inv(cx) < kSerialHot) e |= dm.inv(cx) << (16 + kO1Log);
        else e |= kSerialSlow | cx << 9;
        t.et[blockIdx.x << kO1Log | i] = e;
    }
}

// `groups` times kSerialGroup lookups of wave 0 from the state cur (its entry is E): logs the states whose
// entries it takes, moves the read position p down and counts the escapes in el. kEsc: escapes are taken
// in the entries (SerialMap::esc). All values are the same in every lane; they stay in vector registers
// except for the rare-path test, whose reads of E go to a scalar register under the lookup's latency.
// Cycles a step on a synthetic table without rare entries (2.4 GHz): 76 for the lookup chain alone, 27
// more with escapes, 25 with the rare-path test; a refill of the bit buffer every 4 steps costs 26 a step
// and every 6 steps 17, the escape count kept as an end bit in the sign register (no add a step) saves 9.
template <bool kEsc>
__device__ __forceinline__ void serial_groups(uint32_t& E_, uint32_t& cur_, uint32_t& p_, uint32_t& el_, uint32_t groups,
                                              const FZ_LDS uint32_t* hot, const FZ_LDS uint32_t* ring,
                                              const FZ_LDS uint32_t* signs, FZ_LDS uint32_t* lg,
                                              const FZ_GLB uint32_t* et, const SerialMap& dm) {
    const FZ_LDS uint8_t* lh = reinterpret_cast<const FZ_LDS uint8_t*>(hot);
    uint32_t E = E_, cur = cur_, p = p_, el = el_, sgn = 0, ess = 0;
    asm volatile("" : "+v"(E), "+v"(cur), "+v"(p), "+v"(el));
    uint32_t phase = 0;
    for (uint32_t g = 0; g < groups; g++) {
        // eighteen signs from bit 13 up and an end bit, enough for three groups; the end bit's place
        // tells how many were taken
        if (kEsc && phase == 0) {
            el += g ? (uint32_t)__builtin_clz(sgn) : 0u;
            const FZ_LDS uint32_t* sw = signs + ((el >> 5) & (kSerialSigns - 1));
            sgn = __builtin_amdgcn_alignbit(sw[1], sw[0], el & 31u) << 13 | 1u << 31;
            phase = 3;
        }
        phase--;
        // the 96 bits below the read position: six steps read at most 78
        const FZ_LDS uint32_t* w = ring + (((p - 96u) >> 5) & (kSerialRing - 1));
        const uint32_t w0 = w[0], w1 = w[1], w2 = w[2], w3 = w[3], sh = p & 31u;
        uint64_t buf = (uint64_t)__builtin_amdgcn_alignbit(w3, w2, sh) << 32 | __builtin_amdgcn_alignbit(w2, w1, sh);
        const uint32_t rest = __builtin_amdgcn_alignbit(w1, w0, sh);
        uint32_t w31 = (uint32_t)(buf >> 32) >> 1, sgn13 = kEsc ? sgn & kSerialEsc : 0u;
        asm volatile("" : "+v"(w31), "+v"(sgn13));
        uint32_t states[kSerialGroup];
        uint32_t nbs = 0;
#pragma unroll
        for (int k = 0; k < (int)kSerialGroup; k++) {
            // in issue order: the next lookup, what its latency hides, the rare path
            states[k] = cur;
            const uint32_t Es = __builtin_amdgcn_readfirstlane(E);
            const uint32_t t = w31 >> (E & 31u);
            const uint32_t base = E >> 16;
            uint32_t at = (t + (kEsc ? (sgn13 & E) | base : base)) << 2;
            uint32_t nx = *reinterpret_cast<const FZ_LDS uint32_t*>(lh + at);
            __builtin_amdgcn_sched_barrier(0);
            const uint32_t nb = (E >> 5) & 15u;
            buf <<= nb;
            nbs += nb;
            if (k == 2) buf |= ((uint64_t)rest << 31) >> (63u - nbs);  // at most 39 bits have gone
            w31 = (uint32_t)(buf >> 32) >> 1;
            if (kEsc) {
                sgn >>= (E >> 13) & 1u;
                sgn13 = sgn & kSerialEsc;
            }
            // both ready before the lookup returns (they would be computed where they are used, after it)
            asm volatile("" : "+v"(w31), "+v"(sgn13));
            __builtin_amdgcn_sched_barrier(0);
            if (__builtin_expect((Es & kSerialSlow) != 0, 0)) {
                const uint32_t x = base + t;
                uint32_t c2 = (Es >> 9) & 15u;
                if (!kEsc && c2 == 15u) {  // an escape: its sign from the ring
                    const uint32_t ei = uniform32(el + ess);
                    c2 = 13u + (uniform32(signs[(ei >> 5) & (kSerialSigns - 1)] >> (ei & 31u)) & 1u);
                    ess++;
                    const uint32_t r = dm.inv(c2);
                    if (r < (uint32_t)kSerialHot) {
                        at = (r << kO1Log | x) << 2;
                        nx = *reinterpret_cast<const FZ_LDS uint32_t*>(lh + at);
                        c2 = 15u;
                    }
                }
                if (kEsc || c2 != 15u) {
                    at = kLogCold | (c2 << kO1Log | x) << 2;
                    nx = (et + (c2 << kO1Log))[x];
                }
            }
            cur = at;
            E = nx;
        }
#pragma unroll
        for (int k = 0; k < (int)kSerialGroup; k += 2)
            *reinterpret_cast<FZ_LDS u32x2*>(lg + kSerialGroup * g + k) = u32x2{states[k], states[k + 1]};
        p -= nbs;
    }
    E_ = E;
    cur_ = cur;
    p_ = p;
    el_ = kEsc ? el + (uint32_t)__builtin_clz(sgn) : el + ess;
}

__global__ void __launch_bounds__(kSerialThreads) k_o1d_serial(const SerialJob* jobs) {
    __shared__ uint32_t hot[kSerialHot << kO1Log];
    __shared__ uint32_t ring[kSerialRing + 3];     // word j of the chain at j mod kSerialRing; the first three again at the end
    __shared__ uint32_t signs[kSerialSigns + 1];   // signs of escapes 32 w .. 32 w + 31 at w mod kSerialSigns; likewise
    __shared__ __align__(16) uint32_t log[2][kSerialLog + 4];
    // written by one wave for the others' next round, by the round's parity
    __shared__ uint32_t sh_n[2], sh_fin[2];
    __shared__ uint64_t sh_e[2], sh_done[2];
    __shared__ int64_t sh_a[2];
    const SerialJob& J = jobs[blockIdx.x];
    const uint32_t tid = threadIdx.x, l = tid & 63u, wv = tid >> 6;
    if (J.times && tid == 0) J.times[0] = __builtin_amdgcn_s_memrealtime();
    const SerialMap dm = J.map;
    const uint64_t m = J.m, novf = J.novf;
    const FZ_GLB uint32_t* dt = glb(J.dt);
    const FZ_GLB uint32_t* et = glb(J.et);
    const FZ_GLB int16_t* ov = glb(J.ov);
    const ChainWords cw(J.cb);
    const uint32_t maxc = dm.run + 1;
    {
        u32x4* h = reinterpret_cast<u32x4*>(hot);
        for (uint32_t i = tid; i < (uint32_t)kSerialHot << (kO1Log - 2); i += kSerialThreads)
            h[i] = *reinterpret_cast<const FZ_GLB u32x4*>(et + (dm.perm(i >> (kO1Log - 2)) << kO1Log) +
                                                          4 * (i & ((1u << (kO1Log - 2)) - 1)));
    }
    // stages words [lo, hi) by n lanes of which this is the i-th
    auto stage_words = [&](int64_t lo, int64_t hi, uint32_t i, uint32_t n) {
        for (int64_t j0 = lo; j0 < hi; j0 += 4 * (int64_t)n) {
            uint32_t v[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int64_t j = j0 + q * (int64_t)n + i;
                v[q] = j < hi ? cw.word(j) : 0u;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const int64_t j = j0 + q * (int64_t)n + i;
                const uint32_t r = (uint32_t)j & (kSerialRing - 1);
                if (j < hi) {
                    ring[r] = v[q];
                    if (r < 3) ring[kSerialRing + r] = v[q];
                }
            }
        }
    };
    // stages the signs of escapes [from, to), multiples of 64, by one wave
    auto stage_signs = [&](uint64_t from, uint64_t to) {
        for (uint64_t e = from; e < to; e += 256) {
            int v[4];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint64_t k = e + 64 * q + l;
                v[q] = k < novf ? (int)ov[k] : 0;
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint64_t mk = __ballot(v[q] < 0);
                const uint32_t w = (uint32_t)((e + 64 * q) >> 5) & (kSerialSigns - 1);
                if (l < 2 && e + 64 * q < to) {
                    signs[w + l] = (uint32_t)(mk >> (32 * l));
                    if (w + l == 0) signs[kSerialSigns] = (uint32_t)mk;
                }
            }
        }
    };
    // read positions count from the aligned word that holds the chain's first byte
    constexpr int64_t kRoundBits = 13 * (int64_t)(kSerialLog + 4);
    const int64_t a0 = J.pos0 + cw.shift;
    auto words_for = [&](int64_t a) { return (a - 2 * kRoundBits - 128) >> 5; };
    int64_t staged = words_for(a0);  // words from here up are in the ring
    uint64_t esigns = 4 * 1024 - 64 * 4;
    stage_words(staged, (a0 + 31) >> 5, tid, kSerialThreads);
    if (wv == 2) stage_signs(0, esigns);
    if (tid == 0) {
        sh_n[0] = sh_n[1] = 0;
        sh_fin[0] = sh_fin[1] = 0;
        sh_a[0] = a0;
        sh_e[0] = 0;
        sh_done[0] = 0;
    }
    // wave 0
    int64_t a = a0;
    uint64_t e = 0, steps = 0;        // escapes, entries taken
    uint32_t before = 0;              // entries of the round that is being expanded
    uint32_t cx = 0, X = J.x0 & ((1u << kO1Log) - 1);  // state, where it is not in cur
    uint32_t cur = 0, E = 0;          // log value of the current state, its entry
    bool have = false;                // cur and E hold the state
    // wave 1
    uint64_t done = 0, eo = 0;
    bool bad = false;
    __syncthreads();
    for (uint32_t round = 0;; round++) {
        const uint32_t par = round & 1u;
        if (wv == 0) {
            if (!uniform32(sh_fin[par])) {
                // symbols left for certain: those not expanded yet count as many as they can be
                const uint64_t known = uniform64(sh_done[par]);
                const uint64_t used = known + (uint64_t)maxc * before;
                const uint64_t left = maxc == 1 ? m - steps : used < m ? m - used : 0;
                const uint32_t groups = (uint32_t)min<uint64_t>(kSerialLog / kSerialGroup, left / (kSerialGroup * maxc));
                FZ_LDS uint32_t* lg = lds(log[par]);
                uint32_t n = 0;
                bool fin = false;
                if (groups) {
                    if (!have) {
                        const uint32_t r = dm.inv(cx);
                        cur = r < (uint32_t)kSerialHot ? (r << kO1Log | X) << 2 : kLogCold | (cx << kO1Log | X) << 2;
                        E = et[cx << kO1Log | X];
                        have = true;
                    }
                    uint32_t p = (uint32_t)a;  // wraps: only its place in the ring matters
                    uint32_t el = (uint32_t)e;
                    if (dm.esc) serial_groups<true>(E, cur, p, el, groups, lds(hot), lds(ring), lds(signs), lg, et, dm);
                    else serial_groups<false>(E, cur, p, el, groups, lds(hot), lds(ring), lds(signs), lg, et, dm);
                    n = kSerialGroup * groups;
                    a -= (int64_t)uniform32((uint32_t)a - p);
                    e += uniform32(el - (uint32_t)e);
                } else if (before == 0 || maxc == 1) {
                    // the last few symbols, one step at a time
                    const uint32_t rest = (uint32_t)(maxc == 1 ? m - steps : known < m ? m - known : 0);
                    if (have) {
                        const uint32_t c = uniform32(cur);
                        cx = c & kLogCold ? (c >> (kO1Log + 2)) & 15u : dm.perm(c >> (kO1Log + 2));
                        X = (c >> 2) & ((1u << kO1Log) - 1);
                    }
                    for (; n < rest; n++) {
                        const uint32_t raw = uniform32(dt[cx << kO1Log | X]);
                        lg[n] = kLogSingle | (cx << kO1Log | X) << 2;
                        const uint32_t nb = (raw >> 24) & 15u;
                        a -= nb;
                        const FZ_LDS uint32_t* w = lds(ring) + ((uint32_t)(a >> 5) & (kSerialRing - 1));
                        const uint32_t bits = __builtin_amdgcn_alignbit(w[1], w[0], (uint32_t)a & 31u) & ((1u << nb) - 1u);
                        X = uniform32((raw + bits) & ((1u << kO1Log) - 1));
                        cx = raw >> 28;
                        if (cx == 15u) {
                            cx = 13u + uniform32((lds(signs)[(uint32_t)(e >> 5) & (kSerialSigns - 1)] >> (e & 31u)) & 1u);
                            e++;
                        }
                    }
                    fin = true;
                }
                steps += n;
                before = n;
                if (l == 0) {
                    sh_n[par] = n;
                    sh_fin[par ^ 1u] = fin;
                    sh_a[par ^ 1u] = a;
                    sh_e[par ^ 1u] = e;
                }
            } else if (l == 0) {
                sh_n[par] = 0;
                sh_fin[par ^ 1u] = 2;
            }
        } else if (wv == 1) {
            // expands the round before
            const uint32_t n = uniform32(sh_n[par ^ 1u]);
            const FZ_LDS uint32_t* lg = lds(log[par ^ 1u]);
            FZ_GLB int16_t* out = glb(J.out);
            constexpr int kB = 4;  // states a lane at a time, their table reads in flight together
            for (uint32_t i0 = 0; i0 < n; i0 += 64 * kB) {
                uint32_t raw[kB], last[kB];
                uint8_t cnt[kB], single[kB];
#pragma unroll
                for (int q = 0; q < kB; q++) {
                    const uint32_t i = i0 + 64u * q + l;
                    const uint32_t v = i < n ? lg[i] : 0u;
                    const uint32_t c = v >= kLogCold ? (v >> (kO1Log + 2)) & 15u : dm.perm(v >> (kO1Log + 2));
                    raw[q] = dt[c << kO1Log | ((v >> 2) & ((1u << kO1Log) - 1))];
                    cnt[q] = i < n;
                    single[q] = i >= n || (v & kLogSingle);
                }
                // the symbol an entry ends with, and how many come before it
#pragma unroll
                for (int q = 0; q < kB; q++) last[q] = raw[q];
                for (uint32_t k = 0; k < dm.run; k++) {
                    bool walk = false;
#pragma unroll
                    for (int q = 0; q < kB; q++) {
                        if (cnt[q] == k + 1 && !single[q] && (last[q] >> 24) < 0xF0u && ((last[q] >> 24) & 15u) == 0) {
                            last[q] = dt[last[q] >> 28 << kO1Log | (last[q] & ((1u << kO1Log) - 1))];
                            cnt[q]++;
                            walk = true;
                        }
                    }
                    if (!__ballot(walk)) break;
                }
                // places: counts and escapes of the states before; escaped values
                uint64_t at[kB];
                int code[kB];
#pragma unroll
                for (int q = 0; q < kB; q++) {
                    uint32_t pre = cnt[q];
                    if (dm.run) {
#pragma unroll
                        for (int d = 1; d < 64; d <<= 1) {
                            const uint32_t o = __shfl_up(pre, d);
                            if (l >= (uint32_t)d) pre += o;
                        }
                        at[q] = done + pre - cnt[q];
                        done += uniform32(__shfl(pre, 63));
                    } else {
                        at[q] = done + l;
                        done += (uint32_t)__popcll(__ballot(cnt[q] != 0));
                    }
                    const uint32_t sy = (last[q] >> 16) & 0xFFu;
                    code[q] = (int)((sy >> 1) ^ (~(sy & 1) + 1));
                    const bool esc = cnt[q] && last[q] >> 28 == 15u;
                    const uint64_t em = __ballot(esc);
                    if (esc) {
                        const uint64_t ei = eo + (uint32_t)__popcll(em & ((1ull << l) - 1));
                        code[q] = ei < novf ? (int)ov[ei] : 32767;
                        bad = bad || ei >= novf;
                    }
                    eo += (uint32_t)__popcll(em);
                }
#pragma unroll
                for (int q = 0; q < kB; q++) {
                    if (cnt[q] && at[q] + cnt[q] <= m) {
                        uint32_t rw = raw[q];
                        for (uint32_t k = 1; k < cnt[q]; k++) {
                            const uint32_t sy = (rw >> 16) & 0xFFu;
                            out[at[q]++] = (int16_t)((sy >> 1) ^ (~(sy & 1) + 1));
                            rw = dt[rw >> 28 << kO1Log | (rw & ((1u << kO1Log) - 1))];
                        }
                        out[at[q]] = (int16_t)code[q];
                    } else if (cnt[q]) {
                        bad = true;
                    }
                }
            }
            if (l == 0) sh_done[par ^ 1u] = done;
        } else {
            // two rounds ahead of where wave 0 was when this one began
            const int64_t lo = words_for(uniform64((uint64_t)sh_a[par]));
            if (lo < staged) {
                stage_words(lo, staged, l, 64);
                staged = lo;
            }
            const uint64_t to = (uniform64(sh_e[par]) + 2 * (kSerialLog + 4) + 64 + 63) & ~63ull;
            if (to > esigns) {
                stage_signs(esigns, to);
                esigns = to;
            }
        }
        __syncthreads();
        // the round in which wave 0 had nothing left has expanded the last log; a stream that ran far
        // below its first bit is corrupt
        if (sh_fin[par ^ 1u] == 2) break;
        if (sh_a[par ^ 1u] < -128) {
            bad = true;
            break;
        }
    }
    if (wv == 1) {
        bad = bad || done != m || eo != novf;
        if (__ballot(bad) && l == 0) *J.err = 1;
    } else if (wv == 0 && l == 0 && bad) {
        *J.err = 1;
    }
    if (J.times && tid == 0) J.times[1] = __builtin_amdgcn_s_memrealtime();
}

// ---------------------------------------------------------------- method 0 decode
__device__ inline uint64_t get_msb_field(const uint8_t* buf, uint64_t off, int k) {
    uint64_t v = 0;
    for (int j = 0; j < k; j++) {
        const uint64_t b = off + j;
        v = (v << 1) | ((buf[b >> 3] >> (7 - (b & 7))) & 1u);
    }
    return v;
}

// Escaped codes from their classes and MSB-first mantissas (inverse of escape_streams), one per lane.
__global__ void __launch_bounds__(256) k_ovf_values(const uint8_t* vcl, const uint64_t* voff, const uint8_t* vman,
                                                    uint64_t vman_bits, uint64_t n, int16_t* ovf, int* err) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int k = vcl[i];
    if (k > 16 || voff[i] + (uint64_t)k > vman_bits) {
        *err = 1;
        ovf[i] = 0;
        return;
    }
    const uint64_t vv = (1ull << k) | get_msb_field(vman, voff[i], k);
    const uint32_t zz = (uint32_t)(vv - 1);
    ovf[i] = (int16_t)(int32_t)((zz >> 1) ^ (~(zz & 1) + 1));
}
// Mantissa fields are read only inside the stream's mantissa bytes (rman_bits, vman_bits); a class
// that points past them marks the stream corrupt.
__global__ void k_runs_decode(const uint8_t* rcl, const uint64_t* roff, const uint8_t* rman, uint64_t rman_bits,
                              uint64_t nr, uint64_t* runlen, int* err) {
    const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nr) return;
    const int k = rcl[j];
    if (k > 40 || roff[j] + (uint64_t)k > rman_bits) {
        *err = 1;
        runlen[j] = 0;
        return;
    }
    runlen[j] = ((1ull << k) | get_msb_field(rman, roff[j], k)) - 1;
}
__global__ void k_values_place(const uint8_t* vcl, const uint64_t* voff, const uint8_t* vman, uint64_t vman_bits,
                               uint64_t nv, const uint64_t* runsum, uint64_t n, int16_t* out, int* err) {
    const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nv) return;
    const int k = vcl[j];
    if (k > 17 || voff[j] + (uint64_t)k > vman_bits) {
        *err = 1;
        return;
    }
    const uint64_t vv = (1ull << k) | get_msb_field(vman, voff[j], k);
    const uint32_t zz = (uint32_t)(vv - 1);
    const int32_t f = (int32_t)((zz >> 1) ^ (~(zz & 1) + 1));
    const uint64_t p = runsum[j] + j;  // zeros before value j plus the j values before it
    if (p < n) out[p] = (int16_t)f;
}

struct ToU64 {
    __device__ __forceinline__ uint64_t operator()(const uint8_t& x) const { return x; }
};

struct Add16 {
    __device__ __forceinline__ int16_t operator()(const int16_t& a, const int16_t& b) const { return (int16_t)(a + b); }
};

// ---------------------------------------------------------------- host orchestration
static void sync(hipStream_t st) { FZ_HIP(hipStreamSynchronize(st)); }
template <typename T>
static void d2h(T* h, const T* d, size_t n, hipStream_t st) {
    FZ_HIP(hipMemcpyAsync(h, d, n * sizeof(T), hipMemcpyDeviceToHost, st));
    sync(st);
}
template <typename T>
static void h2d(T* d, const T* h, size_t n, hipStream_t st) {
    FZ_HIP(hipMemcpyAsync(d, h, n * sizeof(T), hipMemcpyHostToDevice, st));
}

// Scratch for cub calls is sized per call from the arena.
static void* cub_scratch(DevArena& ws, size_t bytes) { return ws.take<uint8_t>(bytes ? bytes : 1); }

static void exclusive_scan_u64(const uint64_t* in, uint64_t* out, uint64_t n, DevArena& ws, hipStream_t st) {
    if (n == 0) return;
    size_t bytes = 0;
    FZ_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, (int64_t)n, st));
    void* tmp = cub_scratch(ws, bytes);
    FZ_HIP(hipcub::DeviceScan::ExclusiveSum(tmp, bytes, in, out, (int64_t)n, st));
}

// Every write into the caller's buffer is preceded by a host-side check of its capacity.
static void need_room(uint64_t want, uint64_t cap) {
    if (want > cap) throw std::length_error("The buffer for compressed data is not large enough.");
}

// fse_enc over class-byte arrays (RleFse:150-176), every block of every array in one launch and
// one host round trip for the sizes. Item i writes its framed blocks at out (capacity cap), or,
// with follow set, right after item i - 1's output (in what is left of its capacity); size
// receives the framed length.
struct FseEncItem {
    const uint8_t* src;
    uint64_t n;
    uint8_t* out;
    uint64_t cap;
    bool follow;
    uint64_t size;
};
// Launches the FSE blocks of streams of class bytes (src, length), in their order: block b's framed bytes
// go to slots + b * kFseSlot, their number to sizes[b]. No host round trip.
constexpr uint64_t kFseSlot = kFblk + 1024;
struct FseBlocks {
    std::vector<FseBlk> blks;
    FseBlk* dblks = nullptr;
    uint8_t* slots = nullptr;
    uint64_t* sizes = nullptr;
    void add(const uint8_t* src, uint64_t n) {
        for (uint64_t o = 0; o < n; o += kFblk)
            blks.push_back(FseBlk{src + o, nullptr, (uint32_t)std::min<uint64_t>(kFblk, n - o), 0});
    }
    // blks stays as it is until the stream has been waited for
    void launch(DevArena& ws, hipStream_t st) {
        const uint64_t nb = blks.size();
        if (nb == 0) return;
        slots = ws.take<uint8_t>(nb * kFseSlot);
        sizes = ws.take<uint64_t>(nb);
        dblks = ws.take<FseBlk>(nb);
        FseMeta* meta = ws.take<FseMeta>(nb);
        uint32_t* logs = ws.take<uint32_t>(nb * kFseLogWords);
        h2d(dblks, blks.data(), nb, st);
        uint32_t longest = 0;
        for (const FseBlk& b : blks) longest = std::max(longest, b.len);
        // two chains of up to (longest - 1) / 2 steps, four waves a workgroup
        const unsigned pieces = std::max(1u, ((longest - 1) / 2 + kFsePiece - 1) / kFsePiece);
        FZ_LAUNCH("fse_tables", 0, k_fse_tables, dim3((unsigned)nb), dim3(256), 0, st, dblks, slots, kFseSlot, meta);
        FZ_LAUNCH("fse_sets", 0, k_fse_sets, dim3((unsigned)nb, (pieces + 1) / 2), dim3(256), 0, st, dblks, meta, logs);
        FZ_LAUNCH("fse_finish", 0, k_fse_finish, dim3((unsigned)nb), dim3(256), 0, st, dblks, meta, logs, slots, kFseSlot,
                  sizes);
        FZ_HIP(hipGetLastError());
    }
};

static void fse_enc_multi(std::vector<FseEncItem>& items, DevArena& ws, hipStream_t st) {
    FseBlocks F;
    for (FseEncItem& it : items) {
        it.size = 0;
        F.add(it.src, it.n);
    }
    const uint64_t nb = F.blks.size();
    if (nb == 0) return;
    F.launch(ws, st);
    std::vector<uint64_t> hs(nb);
    d2h(hs.data(), F.sizes, nb, st);
    uint64_t b = 0;
    for (size_t i = 0; i < items.size(); i++) {
        FseEncItem& it = items[i];
        if (it.follow && i > 0) {
            it.out = items[i - 1].out + items[i - 1].size;
            it.cap = items[i - 1].cap - items[i - 1].size;
        }
        uint64_t acc = 0;
        for (uint64_t o = 0; o < it.n; o += kFblk, b++) {
            F.blks[b].dst = it.out + acc;
            acc += hs[b];
        }
        need_room(acc, it.cap);
        it.size = acc;
    }
    h2d(F.dblks, F.blks.data(), nb, st);
    FZ_LAUNCH("fse_pack", 0, k_pack_slots, dim3(64, (unsigned)nb), dim3(256), 0, st, F.slots, kFseSlot, F.sizes, F.dblks);
    FZ_HIP(hipGetLastError());
    sync(st);  // blks is read by the copy above
}

static void put64(uint8_t*& p, uint64_t v) { memcpy(p, &v, 8); p += 8; }

// One part of a stream assembly: len bytes (at most kPieceBytes) from src to dst, device memory.
struct CopyPiece {
    const uint8_t* src;
    uint8_t* dst;
    uint64_t len;
};
constexpr uint64_t kPieceBytes = 64 << 10;
// A workgroup a part; consecutive threads take consecutive bytes, 16 loads in flight per thread.
__global__ void __launch_bounds__(256) k_copy_pieces(const CopyPiece* pieces) {
    const CopyPiece c = pieces[blockIdx.x];
    for (uint64_t i0 = threadIdx.x; i0 < c.len; i0 += 16ull * blockDim.x) {
        uint8_t t[16];
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const uint64_t i = i0 + (uint64_t)k * blockDim.x;
            t[k] = i < c.len ? c.src[i] : (uint8_t)0;
        }
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const uint64_t i = i0 + (uint64_t)k * blockDim.x;
            if (i < c.len) c.dst[i] = t[k];
        }
    }
}

static size_t encode_method0(const int16_t* bins, uint64_t n, uint8_t* out, uint64_t cap, DevArena& ws,
                             hipStream_t st) {
    need_room(48, cap);
    uint64_t* pos = ws.take<uint64_t>(n + 1);
    uint64_t* nsel = ws.take<uint64_t>(1);
    {
        select_indices(bins, n, NonZero{}, pos, nsel, cub_scratch(ws, select_scratch_bytes(n)), "rle_select_values", st);
    }
    uint64_t nv = 0;
    d2h(&nv, nsel, 1, st);
    uint64_t last_pos = 0;
    if (nv) d2h(&last_pos, pos + nv - 1, 1, st);
    const uint64_t nr = (nv == 0) ? 1 : (last_pos == n - 1 ? nv : nv + 1);
    uint8_t* rcl = ws.take<uint8_t>(nr + 1);
    uint8_t* vcl = ws.take<uint8_t>(nv + 1);
    uint64_t* rbits = ws.take<uint64_t>(nr + 1);
    uint64_t* vbits = ws.take<uint64_t>(nv + 1);
    uint64_t* roff = ws.take<uint64_t>(nr + 1);
    uint64_t* voff = ws.take<uint64_t>(nv + 1);
    FZ_LAUNCH("rle_runs_values", n * 2, k_runs_values, dim3(nblk(std::max(nr, nv))), dim3(256), 0, st, bins, n, pos, nv, nr, rcl, vcl,
                       rbits, vbits);
    FZ_HIP(hipGetLastError());
    exclusive_scan_u64(rbits, roff, nr, ws, st);
    exclusive_scan_u64(vbits, voff, nv, ws, st);
    uint64_t rlast[2] = {0, 0}, vlast[2] = {0, 0};
    d2h(&rlast[0], roff + nr - 1, 1, st);
    d2h(&rlast[1], rbits + nr - 1, 1, st);
    if (nv) { d2h(&vlast[0], voff + nv - 1, 1, st); d2h(&vlast[1], vbits + nv - 1, 1, st); }
    const uint64_t rbp = (rlast[0] + rlast[1] + 7) / 8, vbp = nv ? (vlast[0] + vlast[1] + 7) / 8 : 0;
    uint32_t* rman = ws.take<uint32_t>(rbp / 4 + 2);
    uint32_t* vman = ws.take<uint32_t>(vbp / 4 + 2);
    FZ_HIP(hipMemsetAsync(rman, 0, (rbp / 4 + 2) * 4, st));
    FZ_HIP(hipMemsetAsync(vman, 0, (vbp / 4 + 2) * 4, st));
    FZ_LAUNCH("rle_mantissas", 0, k_scatter_mantissas, dim3(nblk(std::max(nr, nv))), dim3(256), 0, st, bins, n, pos, nv, nr, roff,
                       voff, rcl, vcl, rman, vman);
    FZ_HIP(hipGetLastError());
    // class streams go after the 48-byte head
    uint8_t* body = out + 48;
    std::vector<FseEncItem> fe{{rcl, nr, body, cap - 48, false, 0}, {vcl, nv, nullptr, 0, true, 0}};
    fse_enc_multi(fe, ws, st);
    const uint64_t s_rcl = fe[0].size, s_vcl = fe[1].size;
    need_room(48 + s_rcl + s_vcl + rbp + vbp, cap);
    FZ_HIP(hipMemcpyAsync(body + s_rcl + s_vcl, rman, rbp, hipMemcpyDeviceToDevice, st));
    FZ_HIP(hipMemcpyAsync(body + s_rcl + s_vcl + rbp, vman, vbp, hipMemcpyDeviceToDevice, st));
    uint8_t head[48], *p = head;
    put64(p, nr); put64(p, nv); put64(p, s_rcl); put64(p, s_vcl); put64(p, rbp); put64(p, vbp);
    FZ_HIP(hipMemcpyAsync(out, head, 48, hipMemcpyHostToDevice, st));
    sync(st);
    return 48 + s_rcl + s_vcl + rbp + vbp;
}

// Escaped codes of one segment (RleFse:483-532): [u8 0][int16 x n] raw, or, when shorter,
// [u8 1][u64 class bytes][u64 mantissa bytes][class bytes through fse_enc][mantissas], where a
// value's class is k = floor(log2(zigzag + 1)) and its mantissa the k low bits of zigzag + 1, MSB
// first. The values of all segments are one array: tiles of 4,096 (16 values a thread) give classes and
// the bits of a tile, the tiles' sums are scanned, and every thread packs its 16 mantissas into
// whole words. Nothing waits for the host before the coded sizes are read. Segment by segment, with a
// scan of 8-byte bit counts and an atomic for every byte that a mantissa touches, the 15 segments of a
// 512^3 field at 1e-4 (67 million escapes) took 3.9 ms of kernels beside their FSE blocks and a host round trip each,
// all at once take 0.57.
__device__ __forceinline__ uint32_t ovf_zigzag1(int32_t f) { return (((uint32_t)f << 1) ^ (uint32_t)(f >> 31)) + 1u; }
__device__ __forceinline__ uint32_t ovf_class(int32_t f) { return 31u - (uint32_t)__clz((int)ovf_zigzag1(f)); }

// A thread's 16 values from i0 on (0, of class 0, at and past n). ovf is 16-byte aligned.
__device__ __forceinline__ void ovf_load(const int16_t* ovf, uint64_t i0, uint64_t n, int32_t (&f)[16]) {
    if (i0 + 16 <= n) {
        const uint4* p = reinterpret_cast<const uint4*>(ovf + i0);
        const uint4 a = p[0], b = p[1];
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int r = 0; r < 8; r++) {
            f[2 * r] = (int16_t)w[r];
            f[2 * r + 1] = (int16_t)(w[r] >> 16);
        }
    } else {
#pragma unroll
        for (int k = 0; k < 16; k++) f[k] = i0 + k < n ? ovf[i0 + k] : 0;
    }
}

// Exclusive prefix of a thread's v over a workgroup of 256, and the workgroup's sum.
__device__ __forceinline__ uint32_t tile_prefix(uint32_t v, uint32_t* part, uint32_t* sum) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(inc, d, 64);
        if (lane >= d) inc += y;
    }
    if (lane == 63) part[wave] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (uint32_t w = 0; w < 4; w++) {
        before += w < wave ? part[w] : 0u;
        all += part[w];
    }
    *sum = all;
    return before + inc - v;
}

// vcl (16-byte aligned, room for whole tiles): the classes; bits[t]: a tile's mantissa bits (at most 2^16).
__global__ void __launch_bounds__(256) k_ovf_classes(const int16_t* ovf, uint64_t n, uint8_t* vcl, uint32_t* bits) {
    __shared__ uint32_t part[4];
    const uint64_t i0 = (uint64_t)blockIdx.x * kSelTile + threadIdx.x * kSelLane;
    int32_t f[16];
    ovf_load(ovf, i0, n, f);
    uint32_t w[4] = {0, 0, 0, 0}, own = 0, sum;
#pragma unroll
    for (int k = 0; k < 16; k++) {
        const uint32_t c = ovf_class(f[k]);
        own += c;
        w[k >> 2] |= c << (8 * (k & 3));
    }
    *reinterpret_cast<uint4*>(vcl + i0) = make_uint4(w[0], w[1], w[2], w[3]);
    (void)tile_prefix(own, part, &sum);
    if (threadIdx.x == 0) bits[blockIdx.x] = sum;
}

// below[g] = mantissa bits in front of value off[g]; one workgroup a bound.
__global__ void __launch_bounds__(256) k_ovf_bounds(const int16_t* ovf, uint64_t n, const uint64_t* offs, uint64_t ntiles,
                                                    const uint64_t* total, const uint64_t* off, uint64_t* below) {
    __shared__ uint32_t part[4];
    const uint64_t end = min(off[blockIdx.x], n), t = end / kSelTile, i0 = t * kSelTile + threadIdx.x * kSelLane;
    uint32_t own = 0, sum;
    if (i0 < end) {
        int32_t f[16];
        ovf_load(ovf, i0, end, f);
#pragma unroll
        for (int k = 0; k < 16; k++) own += ovf_class(f[k]);
    }
    (void)tile_prefix(own, part, &sum);
    if (threadIdx.x == 0) below[blockIdx.x] = (t < ntiles ? offs[t] : *total) + sum;
}

// Where the segments' values (S + 1 bounds), mantissa bits and mantissa words lie.
struct OvfSegs {
    const uint64_t* off;    // values
    const uint64_t* below;  // bits in front of them
    const uint64_t* word;   // first word of a segment's mantissas
    uint32_t S;
};

// words: all zero. A thread stores the words that only its values reach and adds its part of a shared
// one; a thread whose values lie in two segments starts anew at the bound.
__global__ void __launch_bounds__(256) k_ovf_mantissas(const int16_t* ovf, uint64_t n, const uint64_t* offs, OvfSegs G,
                                                       uint32_t* words) {
    __shared__ uint32_t part[4];
    const uint64_t i0 = (uint64_t)blockIdx.x * kSelTile + threadIdx.x * kSelLane;
    int32_t f[16];
    ovf_load(ovf, i0, n, f);
    uint32_t own = 0, sum;
#pragma unroll
    for (int k = 0; k < 16; k++) own += ovf_class(f[k]);
    uint64_t at = offs[blockIdx.x] + tile_prefix(own, part, &sum);  // bits of all segments in front
    if (i0 >= n) return;
    uint32_t g = 0;
    while (g + 1 < G.S && G.off[g + 1] <= i0) g++;
    uint64_t next = G.off[g + 1];
    uint64_t acc = 0;
    uint32_t have = 0;
    uint32_t* wp = nullptr;
    bool shared_word = true;
    auto start = [&]() {
        const uint64_t bit = at - G.below[g];
        wp = words + G.word[g] + (bit >> 5);
        have = (uint32_t)(bit & 31u);
        acc = 0;
        shared_word = true;
    };
    auto flush = [&]() {
        if (have) atomicOr(wp, __builtin_bswap32((uint32_t)(acc << (32 - have))));
    };
    start();
#pragma unroll
    for (int k = 0; k < 16; k++) {
        if (i0 + k < n) {
            if (i0 + k >= next) {
                flush();
                while (G.off[g + 1] <= i0 + k) g++;
                next = G.off[g + 1];
                start();
            }
            const uint32_t c = ovf_class(f[k]);
            acc = acc << c | (ovf_zigzag1(f[k]) & ((1u << c) - 1u));
            have += c;
            at += c;
            if (have >= 32) {
                have -= 32;
                const uint32_t w = __builtin_bswap32((uint32_t)(acc >> have));
                if (shared_word) atomicOr(wp, w);
                else *wp = w;
                shared_word = false;
                wp++;
                acc &= (1ull << have) - 1;
            }
        }
    }
    flush();
}

// One segment's escape block: its first bytes, made on the host, then the device bytes that follow.
struct EscapeBlock {
    std::vector<uint8_t> head;
    std::vector<std::pair<const uint8_t*, uint64_t>> parts;
    uint64_t len = 0;
};
// First words of the segments' mantissas at 16 bits a value, the most there are.
static std::vector<uint64_t> escape_words(const std::vector<uint64_t>& off, uint64_t S) {
    std::vector<uint64_t> w(S + 1, 0);
    for (uint64_t g = 0; g < S; g++) w[g + 1] = w[g] + (off[g + 1] - off[g] + 1) / 2 + 1;
    return w;
}
static uint64_t escape_tiles(uint64_t n) { return (n + kSelTile - 1) / kSelTile; }

static void escape_streams(const int16_t* ovf, const std::vector<uint64_t>& off, uint64_t S,
                           std::vector<EscapeBlock>& block, DevArena& ws, hipStream_t st) {
    const uint64_t n = off[S], nt = escape_tiles(n);
    std::vector<uint64_t> hb(S + 1, 0), hs;
    FseBlocks F;
    uint32_t* man = nullptr;
    const std::vector<uint64_t> word = escape_words(off, S);
    if (n) {
        uint8_t* vcl = ws.take<uint8_t>(nt * kSelTile);
        uint32_t* bits = ws.take<uint32_t>(nt);
        uint64_t* offs = ws.take<uint64_t>(nt);
        uint64_t* bounds = ws.take<uint64_t>(3 * (S + 1) + 1);  // value bounds, words, bit bounds, all bits
        uint64_t *doff = bounds, *dword = bounds + S + 1, *dbelow = bounds + 2 * (S + 1), *total = bounds + 3 * (S + 1);
        man = ws.take<uint32_t>(word[S]);
        FZ_HIP(hipMemsetAsync(man, 0, word[S] * 4, st));
        h2d(doff, off.data(), S + 1, st);
        h2d(dword, word.data(), S + 1, st);
        FZ_LAUNCH("o1_escape_classes", n * 3, k_ovf_classes, dim3((unsigned)nt), dim3(256), 0, st, ovf, n, vcl, bits);
        FZ_LAUNCH("o1_escape_bits", nt * 12, k_sel_scan, dim3(1), dim3(1024), 0, st, bits, nt, offs, total);
        FZ_LAUNCH("o1_escape_bits", 0, k_ovf_bounds, dim3((unsigned)(S + 1)), dim3(256), 0, st, ovf, n, offs, nt, total,
                  doff, dbelow);
        FZ_LAUNCH("o1_escape_mantissas", n * 3, k_ovf_mantissas, dim3((unsigned)nt), dim3(256), 0, st, ovf, n, offs,
                  OvfSegs{doff, dbelow, dword, (uint32_t)S}, man);
        FZ_HIP(hipGetLastError());
        // every segment's class bytes through FSE in one launch
        for (uint64_t g = 0; g < S; g++) F.add(vcl + off[g], off[g + 1] - off[g]);
        F.launch(ws, st);
        hs.resize(F.blks.size());
        FZ_HIP(hipMemcpyAsync(hb.data(), dbelow, (S + 1) * 8, hipMemcpyDeviceToHost, st));
        d2h(hs.data(), F.sizes, hs.size(), st);
    }
    uint64_t b = 0;
    for (uint64_t g = 0; g < S; g++) {
        const uint64_t lo = off[g], m = off[g + 1] - lo, raw = 2 * m, vbp = (hb[g + 1] - hb[g] + 7) / 8;
        EscapeBlock& B = block[g];
        uint64_t svcl = 0;
        for (uint64_t o = 0; o < m; o += kFblk, b++) {
            B.parts.push_back({F.slots + b * kFseSlot, hs[b]});
            svcl += hs[b];
        }
        if (m == 0 || svcl + vbp + 16 >= raw) {
            B.head.assign(1, 0);
            B.parts.assign(1, {reinterpret_cast<const uint8_t*>(ovf + lo), raw});
            B.len = 1 + raw;
            continue;
        }
        B.parts.push_back({reinterpret_cast<const uint8_t*>(man + word[g]), vbp});
        B.head.resize(17);
        uint8_t* h = B.head.data();
        *h++ = 1;
        put64(h, svcl);
        put64(h, vbp);
        B.len = 17 + svcl + vbp;
    }
}

// An upper bound of the device workspace escape_streams takes for n escaped values in the
// segments bounded by off (every take rounded up to 256 bytes).
static size_t escape_workspace_bound(const std::vector<uint64_t>& off, uint64_t S) {
    const uint64_t n = off[S], nt = escape_tiles(n);
    size_t bytes = 0;
    auto add = [&](size_t b) { bytes += (b + 255) & ~size_t(255); };
    add(nt * kSelTile);
    add(4 * nt);
    add(8 * nt);
    add(8 * (3 * (S + 1) + 1));
    add(4 * escape_words(off, S)[S]);
    uint64_t nb = 0;
    for (uint64_t g = 0; g < S; g++) nb += (off[g + 1] - off[g] + kFblk - 1) / kFblk;
    add(nb * kFseSlot);
    add(8 * nb);
    add(sizeof(FseBlk) * nb);
    add(sizeof(FseMeta) * nb);
    add(4 * nb * kFseLogWords);
    return bytes + (1u << 16);
}

// escape_streams on the second stream, driven by a helper thread (its layout takes host round
// trips) with a workspace of its own carved out of the call's; joined, and its error rethrown,
// before the encoder output is assembled.
struct EscapeWorker {
    std::thread th;
    std::exception_ptr err;
    DevArena sub;
    ~EscapeWorker() {
        if (th.joinable()) th.join();
    }
    void join() {
        if (th.joinable()) th.join();
        if (err) std::rethrow_exception(err);
    }
};

static size_t encode_method1(const int16_t* bins, uint64_t n, uint8_t* out, uint64_t cap, DevArena& ws,
                             hipStream_t st, const AuxStream& aux) {
    // the piece kernels read the codes in aligned 16-byte loads (arena allocations are 256-byte
    // aligned and rounded up to 256 bytes)
    if (((uintptr_t)bins & 15u) != 0) throw std::logic_error("order-1 encode: codes not 16-byte aligned");
    uint64_t S = n / kO1Seg;
    if (S < 1) S = 1;
    if (S > 16) S = 16;
    const uint64_t seg = (n + S - 1) / S;
    // escaped codes (sym 255) of the whole array, in index order
    int16_t* ovf = ws.take<int16_t>(n + 1);
    uint64_t* nsel = ws.take<uint64_t>(1);
    const SelTiles esc_tiles = select_codes(bins, n, IsO1Escape{}, CopyCode{bins, ovf}, nsel,
                                            cub_scratch(ws, select_scratch_bytes(n)), "o1_select_escapes", st);
    // histograms and tables per segment
    uint32_t* cnt = ws.take<uint32_t>(S * kO1Ctx * kO1Sym);
    uint16_t* nf = ws.take<uint16_t>(S * kO1Ctx * kO1Sym);
    CTable* ct = ws.take<CTable>(S * kO1Ctx);
    uint32_t* use = ws.take<uint32_t>(S * kO1Ctx);
    FZ_HIP(hipMemsetAsync(cnt, 0, S * kO1Ctx * kO1Sym * 4, st));
    std::vector<uint64_t> chains;  // {seg lo, chunk lo, chunk hi, segment}
    std::vector<uint64_t> novf(S * kO1K), ovf_off(S + 1);
    std::vector<uint64_t> seg_n(S), ends;
    uint64_t e = 0;
    // segments of 2^20 codes or more are sampled, in one launch (they are the first ones: every
    // segment but the last is seg long)
    uint64_t s_sampled = 0, nw_max = 0, sampled_codes = 0;
    for (uint64_t g = 0; g < S; g++) {
        const uint64_t lo = g * seg, hi = std::min(lo + seg, n), sn = hi - lo;
        seg_n[g] = sn;
        const uint64_t cs = (sn + kO1K - 1) / kO1K;
        const int16_t* sb = bins + lo;
        uint32_t* c = cnt + g * kO1Ctx * kO1Sym;
        if (sn < (1u << 20)) {
            FZ_LAUNCH("o1_hist", sn * 2, k_o1_hist_exact, dim3(std::min<uint64_t>(1024, nblk(sn))), dim3(256), 0, st, sb, sn, cs, c);
        } else {
            if (s_sampled != g) throw std::logic_error("order-1 histogram: sampled segments out of order");
            const uint64_t step = std::max<uint64_t>(sn / 2048, 512);
            const uint64_t nw = (sn + step - 1) / step;
            nw_max = std::max(nw_max, nw);
            sampled_codes += nw * 512;
            s_sampled = g + 1;
        }
        FZ_HIP(hipGetLastError());
        for (int k = 0; k < kO1K; k++) {
            const uint64_t clo = lo + k * cs, chi = std::min(clo + cs, hi);
            chains.insert(chains.end(), {lo, clo, std::max(chi, clo), g});
            ends.push_back(chi);  // below clo for the empty chunks at the end of a short segment
        }
    }
    if (s_sampled) {
        // about 1,024 workgroups in all
        const uint64_t per = std::max<uint64_t>(1, nw_max * s_sampled / 1024);
        FZ_LAUNCH("o1_hist", sampled_codes * 2, k_o1_hist_sample, dim3((unsigned)((nw_max + per - 1) / per), (unsigned)s_sampled),
                  dim3(256), 0,
                  st, bins, n, seg, (uint64_t)512, cnt);
        FZ_LAUNCH("o1_hist", 0, k_add_one, dim3(nblk(s_sampled * kO1Ctx * kO1Sym)), dim3(256), 0, st, cnt,
                  (int)(s_sampled * kO1Ctx * kO1Sym));
        FZ_HIP(hipGetLastError());
    }
    // escapes below each chain's end
    const int nch = (int)(S * kO1K);
    uint64_t* dends = ws.take<uint64_t>(nch);
    uint64_t* dbelow = ws.take<uint64_t>(nch);
    h2d(dends, ends.data(), nch, st);
    FZ_LAUNCH("o1_escape_counts", 0, k_sel_below<IsO1Escape>, dim3((unsigned)nch), dim3(256), 0, st, bins, n, IsO1Escape{},
              esc_tiles.offs, esc_tiles.count, nsel, dends, dbelow);
    FZ_HIP(hipGetLastError());
    if (aux.stream) {
        FZ_HIP(hipEventRecord(aux.fork, st));
        FZ_HIP(hipStreamWaitEvent(aux.stream, aux.fork, 0));
    }
    // The escape side streams need only the escaped values and their segment offsets: with a second
    // stream they are coded there, beside the chains. Their counts are read over that stream, and only after
    // the chains' first kernels are queued: the main stream has work meanwhile.
    std::vector<EscapeBlock> oblock(S);
    EscapeWorker ew;
    bool counted = false;
    auto start_escapes = [&]() {
        if (counted) return;
        counted = true;
        std::vector<uint64_t> below(nch);
        d2h(below.data(), dbelow, nch, aux.stream ? aux.stream : st);
        for (uint64_t g = 0; g < S; g++) {
            ovf_off[g] = e;
            for (int k = 0; k < kO1K; k++) {
                const int q = (int)(g * kO1K + k);
                const uint64_t clo = chains[4 * q + 1], chi = ends[q];
                const uint64_t b = std::max(below[q], e);
                novf[q] = (chi > clo) ? b - e : 0;
                e = b;
            }
        }
        ovf_off[S] = e;
        if (!aux.stream) return;
        const size_t need = escape_workspace_bound(ovf_off, S);
        ew.sub.bind(ws.take<uint8_t>(need), need);
        int dev = 0;
        FZ_HIP(hipGetDevice(&dev));
        LaunchProfiler* prof = g_prof;
        ew.th = std::thread([&ew, &ovf, &ovf_off, &oblock, &aux, S, dev, prof]() {
            try {
                FZ_HIP(hipSetDevice(dev));
                g_prof = prof;
                escape_streams(ovf, ovf_off, S, oblock, ew.sub, aux.stream);
            } catch (...) {
                ew.err = std::current_exception();
            }
            g_prof = nullptr;
        });
    };
    FZ_LAUNCH("o1_tables", 0, k_o1_tables, dim3(kO1Ctx, (unsigned)S), dim3(256), 0, st, cnt, nf, ct, use);
    FZ_HIP(hipGetLastError());
    uint64_t* dchains = ws.take<uint64_t>(chains.size());
    h2d(dchains, chains.data(), chains.size(), st);
    uint64_t maxcs = 0;
    for (uint64_t g = 0; g < S; g++) maxcs = std::max(maxcs, (seg_n[g] + kO1K - 1) / kO1K);
    // chain staging: 13 bits per symbol at most, plus the closing state; every chain's words start
    // 64-byte aligned (k_o1_emit stores whole aligned 32-byte runs)
    const uint64_t stride_words = ((maxcs * 2 + 4096 + 3) / 4 + 15) & ~(uint64_t)15;
    const uint64_t bstride = stride_words * 4;
    uint32_t* words = ws.take<uint32_t>(nch * stride_words);
    uint8_t* bufs = reinterpret_cast<uint8_t*>(words);
    uint64_t* blen = ws.take<uint64_t>(nch + 1);  // lengths of the chains, and whether their sets failed
    uint64_t* chain_bits = ws.take<uint64_t>(nch);
    // The pieces of every chain (steps i = hi-2 .. lo), laid out on the host; the vector stays until the
    // stream has been waited for.
    auto lay_out = [&](uint32_t steps_piece, std::vector<uint64_t>& pfirst) {
        pfirst.assign(nch + 1, 0);
        for (int q = 0; q < nch; q++) {
            const uint64_t clo = chains[4 * q + 1], chi = chains[4 * q + 2];
            const uint64_t steps = (chi > clo + 1) ? chi - clo - 1 : 0;
            pfirst[q + 1] = pfirst[q] + (steps + steps_piece - 1) / steps_piece;
        }
        uint64_t* dpfirst = ws.take<uint64_t>(nch + 1);
        h2d(dpfirst, pfirst.data(), nch + 1, st);
        return O1Chains{dchains, dpfirst, nch, steps_piece};
    };
    // workgroups a segment in a launch of one lane a piece
    auto groups_of = [&](const std::vector<uint64_t>& first, uint32_t threads) {
        uint64_t most = 1;
        for (uint64_t g = 0; g < S; g++) most = std::max(most, first[(g + 1) * kO1K] - first[g * kO1K]);
        return (uint32_t)((most + threads - 1) / threads);
    };
    std::vector<uint64_t> sets_first, pfirst;
    const bool sets = n <= kSetMaxCodes;
    uint64_t* failed = blen + nch;
    if (sets) {
        const O1Chains CH = lay_out(kSetPiece, sets_first);
        const uint64_t np = sets_first[nch];
        uint64_t most = 0;
        for (int q = 0; q < nch; q++) most = std::max(most, sets_first[q + 1] - sets_first[q]);
        O1Sets B{ws.take<uint16_t>(np * kSetStates + 1), ws.take<uint16_t>(np * kSetStates + 1),
                 ws.take<uint16_t>(np * kSetStates + 1), ws.take<uint8_t>(np + 1)};
        uint32_t* end_state = ws.take<uint32_t>(np + 1);
        uint64_t* bitoff = ws.take<uint64_t>(np + 1);
        FZ_HIP(hipMemsetAsync(failed, 0, sizeof(uint64_t), st));
        if (np)
            FZ_LAUNCH("o1_encode_sets", n * 4, k_o1_sets, dim3((unsigned)((np + 3) / 4)), dim3(256), 0, st, bins, CH, np, ct, nf,
                      B, failed);
        FZ_LAUNCH("o1_encode_walk", 0, k_o1_sets_walk, dim3((unsigned)nch), dim3(256), most * (kSetStates + 1), st, CH, B,
                  end_state, bitoff, chain_bits, words, stride_words, failed);
        if (np)
            FZ_LAUNCH("o1_encode_emit", n * 2, k_o1_emit, dim3((unsigned)S * groups_of(sets_first, kEmitThreads)),
                      dim3(kEmitThreads), 0, st, bins, CH, groups_of(sets_first, kEmitThreads), ct, use, end_state, bitoff, words,
                      stride_words, failed);
        FZ_LAUNCH("o1_encode_close", 0, k_o1_close, dim3(nblk(nch, 64)), dim3(64), 0, st, bins, CH, ct, end_state, chain_bits,
                  words, stride_words, blen, failed);
        FZ_HIP(hipGetLastError());
        start_escapes();
    }
    auto guess_and_repair = [&]() {
        // one round of workgroups of one a CU, whole ones for every segment
        constexpr uint64_t kCus = 256;
        const uint64_t lanes = std::max<uint64_t>(1, kCus / S) * kEncThreads - kO1K;  // a chain's last piece is a part
        const uint32_t steps_piece = (uint32_t)std::min<uint64_t>(kO1Piece, std::max<uint64_t>(kO1PieceMin, ((seg + lanes - 1) / lanes + 15) & ~15ull));
        const O1Chains CH = lay_out(steps_piece, pfirst);
        const uint64_t np = pfirst[nch];
        const uint32_t groups = groups_of(pfirst, kEncThreads);
        uint16_t* slog = ws.take<uint16_t>(np * steps_piece + 16);  // step-major: [step in piece][piece]
        uint32_t* spec_end = ws.take<uint32_t>(np + 1);
        uint32_t* end_a = ws.take<uint32_t>(np + 1);
        uint32_t* end_b = ws.take<uint32_t>(np + 1);
        uint64_t* spec_bits = ws.take<uint64_t>(np + 1);
        uint64_t* nbits = ws.take<uint64_t>(np + 1);
        uint8_t* chg_a = ws.take<uint8_t>(np + 1);
        uint8_t* chg_b = ws.take<uint8_t>(np + 1);
        unsigned int* any = ws.take<unsigned int>(1);
        uint64_t* scan = ws.take<uint64_t>(np + 1);
        uint64_t* bitoff = ws.take<uint64_t>(np + 1);
        if (np) {
            FZ_LAUNCH("o1_encode_spec", n * 4, k_o1_spec, dim3((unsigned)S * groups), dim3(kEncThreads), 0, st, bins, CH, groups, np,
                      ct, use, slog, spec_end, spec_bits);
            FZ_HIP(hipGetLastError());
            start_escapes();
            FZ_HIP(hipMemcpyAsync(nbits, spec_bits, np * 8, hipMemcpyDeviceToDevice, st));
            // fix-up rounds; each round finalizes at least the next piece of every chain, so the loop
            // ends within max-pieces-per-chain rounds
            const uint32_t* end_prev = spec_end;
            uint32_t* end_next = end_a;
            const uint8_t* chg_prev = nullptr;
            uint8_t* chg_next = chg_a;
            uint64_t max_rounds = 1;
            for (int q = 0; q < nch; q++) max_rounds = std::max<uint64_t>(max_rounds, pfirst[q + 1] - pfirst[q] + 1);
            // Two rounds per host check: `any` counts the changes of the second only. A round after one
            // with no change re-runs no piece and changes nothing, so the check ends the loop at the
            // first pair whose second round saw no change.
            for (uint64_t round = 0;;) {
                if (round > max_rounds + 1) throw std::runtime_error("tANS piece fix-up did not settle");
                for (int k = 0; k < 2; k++, round++) {
                    if (k == 1) FZ_HIP(hipMemsetAsync(any, 0, sizeof(unsigned int), st));
                    FZ_LAUNCH("o1_encode_fix", 0, k_o1_fix, dim3((unsigned)S * groups), dim3(kEncThreads), 0, st, bins, CH, groups, np, ct,
                              use, slog, spec_end, spec_bits, end_prev, end_next, nbits, chg_prev, chg_next, any);
                    FZ_HIP(hipGetLastError());
                    end_prev = end_next;
                    end_next = (end_next == end_a) ? end_b : end_a;
                    chg_prev = chg_next;
                    chg_next = (chg_next == chg_a) ? chg_b : chg_a;
                }
                unsigned int h_any = 0;
                d2h(&h_any, any, 1, st);
                if (!h_any) break;
            }
            exclusive_scan_u64(nbits, scan, np, ws, st);
            FZ_LAUNCH("o1_encode_offsets", 0, k_o1_offsets, dim3(nblk(np + nch)), dim3(256), 0, st, CH, np, scan, nbits, bitoff,
                               chain_bits);
            FZ_HIP(hipGetLastError());
            FZ_LAUNCH("o1_encode_clear", 0, k_o1_clear_shared, dim3(nblk(np + nch)), dim3(256), 0, st, CH, np, bitoff, chain_bits,
                               words, stride_words);
            FZ_HIP(hipGetLastError());
            FZ_LAUNCH("o1_encode_emit", n * 2, k_o1_emit, dim3((unsigned)S * groups_of(pfirst, kEmitThreads)), dim3(kEmitThreads), 0,
                      st, bins, CH, groups_of(pfirst, kEmitThreads), ct, use, end_prev, bitoff, words, stride_words,
                      (const uint64_t*)nullptr);
            FZ_HIP(hipGetLastError());
            FZ_LAUNCH("o1_encode_close", 0, k_o1_close, dim3(nblk(nch, 64)), dim3(64), 0, st, bins, CH, ct, end_prev, chain_bits,
                               words, stride_words, blen, (const uint64_t*)nullptr);
        } else {
            FZ_HIP(hipMemsetAsync(chain_bits, 0, nch * 8, st));
            FZ_LAUNCH("o1_encode_clear", 0, k_o1_clear_shared, dim3(nblk(nch)), dim3(256), 0, st, CH, np, bitoff, chain_bits, words,
                               stride_words);
            FZ_HIP(hipGetLastError());
            FZ_LAUNCH("o1_encode_close", 0, k_o1_close, dim3(nblk(nch, 64)), dim3(64), 0, st, bins, CH, ct, spec_end, chain_bits,
                               words, stride_words, blen, (const uint64_t*)nullptr);
        }
        FZ_HIP(hipGetLastError());
    };
    if (!sets) guess_and_repair();
    start_escapes();  // no chain has a step
    // escape side streams, one block per segment
    if (aux.stream) ew.join();
    else escape_streams(ovf, ovf_off, S, oblock, ws, st);
    std::vector<uint64_t> hblen(nch + 1);
    d2h(hblen.data(), blen, nch + (sets ? 1 : 0), st);
    if (sets && hblen[nch]) {  // symbols too frequent or too flat for sets: nothing has been written yet
        guess_and_repair();
        d2h(hblen.data(), blen, nch, st);
    }
    // assemble: [u64 S] then per segment [n][K][blen x4][novf x4][nf][streams][ovf block]
    uint64_t total = 8;
    for (uint64_t g = 0; g < S; g++) {
        total += 8 * 10 + kO1Ctx * kO1Sym * 2 + oblock[g].len;
        for (int k = 0; k < kO1K; k++) total += hblen[g * kO1K + k];
    }
    need_room(total, cap);
    // The headers go to the device in one copy; then one launch moves every piece (headers, tables,
    // chain streams, escape blocks) to its place, in parts of at most kPieceBytes.
    constexpr uint64_t kSegHead = 80 + 17;  // a segment's numbers, its escape block's first bytes
    std::vector<uint8_t> heads(8 + S * kSegHead);
    {
        uint8_t* h = heads.data();
        put64(h, S);
        for (uint64_t g = 0; g < S; g++) {
            h = heads.data() + 8 + g * kSegHead;
            put64(h, seg_n[g]);
            put64(h, kO1K);
            for (int k = 0; k < kO1K; k++) put64(h, hblen[g * kO1K + k]);
            for (int k = 0; k < kO1K; k++) put64(h, novf[g * kO1K + k]);
            memcpy(h, oblock[g].head.data(), oblock[g].head.size());
        }
    }
    uint8_t* dheads = ws.take<uint8_t>(heads.size());
    h2d(dheads, heads.data(), heads.size(), st);
    std::vector<CopyPiece> pieces;
    uint8_t* p = out;
    auto piece = [&](const uint8_t* src, uint64_t len) {
        for (uint64_t o = 0; o < len; o += kPieceBytes)
            pieces.push_back(CopyPiece{src + o, p + o, std::min<uint64_t>(kPieceBytes, len - o)});
        p += len;
    };
    piece(dheads, 8);
    for (uint64_t g = 0; g < S; g++) {
        piece(dheads + 8 + g * kSegHead, 80);
        piece(reinterpret_cast<const uint8_t*>(nf + g * kO1Ctx * kO1Sym), kO1Ctx * kO1Sym * 2);
        for (int k = 0; k < kO1K; k++) {
            const uint64_t q = g * kO1K + k;
            piece(bufs + q * bstride, hblen[q]);
        }
        piece(dheads + 8 + g * kSegHead + 80, oblock[g].head.size());
        for (const auto& part : oblock[g].parts) piece(part.first, part.second);
    }
    CopyPiece* dpieces = ws.take<CopyPiece>(pieces.size());
    h2d(dpieces, pieces.data(), pieces.size(), st);
    FZ_LAUNCH("o1_assemble", 2 * (p - out), k_copy_pieces, dim3((unsigned)pieces.size()), dim3(256), 0, st, dpieces);
    FZ_HIP(hipGetLastError());
    sync(st);  // heads and pieces (host) are read by the copies above
    return (size_t)(p - out);
}

size_t entropy_encode(const int16_t* codes, uint64_t n, uint8_t* out, size_t out_cap, DevArena& ws, hipStream_t st,
                      EntropyStats* stats, const AuxStream& aux) {
    need_room(5, out_cap);
    // preprocess_encode: 256 windows of 32 codes (RleFse:850-895)
    uint64_t NW = 256, WL = 32;
    if (n < NW * WL) { WL = n / NW; if (!WL) WL = 1; }
    uint64_t step = (n > NW * WL) ? (n - WL) / NW : WL;
    if (!step) step = 1;
    PreCounts* pc = ws.take<PreCounts>(1);
    FZ_LAUNCH("preprocess", 0, k_preprocess, dim3(1), dim3(256), 0, st, codes, n, NW, WL, step, pc);
    FZ_HIP(hipGetLastError());
    PreCounts h{};
    d2h(&h, pc, 1, st);
    const double p0 = h.cnt ? 1.0 * (double)h.z / (double)h.cnt : 1.0;
    const double dz = (h.cnt && h.cntd) ? (1.0 * (double)h.zd / (double)h.cntd - p0) : 0.0;
    const int use_delta = dz > 0.005;
    int method = (p0 >= 0.80) ? 0 : 1;
    if (n < (uint64_t)20 * kO1Ctx * kO1Sym) method = 0;
    if (stats) { stats->method = method; stats->use_delta = use_delta; }
    const uint8_t save[5] = {(uint8_t)(method | (use_delta ? 0x80 : 0)), 0, 0, 0, 0};
    FZ_HIP(hipMemcpyAsync(out, save, 5, hipMemcpyHostToDevice, st));  // save lives until the encoders have waited
    const int16_t* bins = codes;
    if (use_delta && n > 0) {
        int16_t* d = ws.take<int16_t>(n);
        FZ_LAUNCH("delta", n * 4, k_delta, dim3(nblk(n)), dim3(256), 0, st, codes, d, n);
        FZ_HIP(hipGetLastError());
        bins = d;
    }
    const size_t body = (method == 1) ? encode_method1(bins, n, out + 5, out_cap - 5, ws, st, aux)
                                      : encode_method0(bins, n, out + 5, out_cap - 5, ws, st);
    return 5 + body;
}

static uint64_t get64(const uint8_t*& p) {
    uint64_t v;
    memcpy(&v, p, 8);
    p += 8;
    return v;
}

// Block offsets of a framed class-byte stream of n bytes (RleFse:150-176: per 64 K block [0][raw],
// [2][symbol] or [1][u32 len][FSE_compress output]), found by walking the block headers within the
// stream's avail bytes. Returns the stream's length; a header or block past avail, or an unknown
// flag, is a corrupt stream.
static uint64_t frame_offsets(const uint8_t* h, uint64_t n, uint64_t avail, std::vector<uint64_t>& offs) {
    uint64_t rp = 0, dp = 0;
    offs.clear();
    auto corrupt = [] { throw std::invalid_argument("corrupt entropy stream: FSE block framing"); };
    while (dp < n) {
        const uint64_t len = std::min<uint64_t>(kFblk, n - dp);
        offs.push_back(rp);
        if (rp >= avail) corrupt();
        const uint8_t flag = h[rp];
        uint64_t blk;
        if (flag == 0) {
            blk = 1 + len;
        } else if (flag == 2) {
            blk = 2;
        } else if (flag == 1) {
            if (avail - rp < 5) corrupt();
            uint32_t rr;
            memcpy(&rr, h + rp + 1, 4);
            if (rr < 2 || rr >= len) corrupt();  // FSE_compress output of a block is shorter than the block
            blk = 5 + (uint64_t)rr;
        } else {
            corrupt();
        }
        if (avail - rp < blk) corrupt();
        rp += blk;
        dp += len;
    }
    return rp;
}

// Decodes framed class-byte streams (host copy hsrc for the block headers, device copy dsrc) of n
// bytes each into out, every block of every stream in one launch.
struct FseDecItem {
    const uint8_t* hsrc;
    const uint8_t* dsrc;
    uint64_t n;
    uint64_t avail;  // bytes of the framed stream
    uint8_t* out;
};
// Appends the blocks of the items; returns whether one of them is FSE-coded with a table log above
// 11 (its NCount header's first four bits hold the log minus 5), which the decoder's big layout
// takes.
static bool fse_block_list(const std::vector<FseDecItem>& items, std::vector<FseBlk>& blks) {
    std::vector<uint64_t> offs;
    bool big = false;
    for (const FseDecItem& it : items) {
        if (it.n == 0) continue;
        // the block decoder stores four symbols at a time (blocks start 64 KiB apart in out)
        if (((uintptr_t)it.out & 3u) != 0) throw std::logic_error("FSE block decode: output not 4-byte aligned");
        frame_offsets(it.hsrc, it.n, it.avail, offs);
        for (size_t k = 0; k < offs.size(); k++) {
            const uint8_t* h = it.hsrc + offs[k];  // an FSE block holds at least 5 + 2 bytes
            if (h[0] == 1 && (h[5] & 0xFu) + kFseMinTableLog > kFblkLog) big = true;
            blks.push_back(FseBlk{it.dsrc + offs[k], it.out + k * kFblk,
                                  (uint32_t)std::min<uint64_t>(kFblk, it.n - k * kFblk), 0});
        }
    }
    return big;
}
static void launch_fse_dec(bool big, const FseBlk* dblks, size_t nb, int* err, hipStream_t st) {
    if (big)
        FZ_LAUNCH("fse_dec_blocks", 0, k_fse_dec_blocks<true>, dim3((unsigned)nb), dim3(256), 0, st, dblks, err);
    else
        FZ_LAUNCH("fse_dec_blocks", 0, k_fse_dec_blocks<false>, dim3((unsigned)nb), dim3(256), 0, st, dblks, err);
}
static void fse_dec_multi(const std::vector<FseDecItem>& items, int* err, DevArena& ws, hipStream_t st) {
    std::vector<FseBlk> blks;
    const bool big = fse_block_list(items, blks);
    if (blks.empty()) return;
    FseBlk* dblks = ws.take<FseBlk>(blks.size());
    h2d(dblks, blks.data(), blks.size(), st);
    launch_fse_dec(big, dblks, blks.size(), err, st);
    FZ_HIP(hipGetLastError());
    sync(st);  // blks is read by the copy above
}

// Order-1 tANS chains are given as 7 values each: stream offset, bytes, out lo, out hi, escape offset,
// table set, escape count.
// Sequential chains of fewer take several steps a lookup (kSerialRun).
constexpr double kSerialRunBits = 2.0;
// In the batched decompress, chains of at most this many are handed to the batch, whose split chains run
// in one set of launches, and whose other chains in one launch beside them: a field's own launches
// leave most of the chip idle (192 chunks of 540,000 codes at bounds 1e-2 to 1e-4: 64 ms with all of
// their chains decoded from their starts, 47 ms like this). So are longer ones that their item's
// region has no room for. The split chains of a batch share at most kBatchSplitBytes of sets and
// graphs, and a quarter of the device memory that is free; chains past that are decoded from their start.
constexpr uint64_t kDeferSymbols = 1ull << 19;
constexpr double kBatchSplitBytes = 4.0 * (1ull << 30);
// Alone, a chain of few bits a symbol runs 64 decoders 2,048 symbols ahead of every part in what the chip
// has to spare. In a batch those steps are what the whole takes (256 of a lane a symbol, as many as L2
// serves in 1.6 ns: 25 of 60 ms for the chunks above), so it runs 32 decoders 1,024 ahead, and the walk
// decodes the few parts more that then lack their entry: 60 -> 49 ms.
constexpr uint32_t kBatchWarm = 32 * 1024;

// Stationary distribution of segment g's context chain (a code's context follows from the previous
// code; an escape leads to 13 or 14, counted half each), from the normalized counts of its 15
// tables at nf_off. Counts of 1 and below (and the low-probability mark -1) are left out: the
// encoder's sampled histograms add one to every symbol, and that floor, spread over the 232
// symbols whose context is 13 or 14, would rank those two contexts far above their use (8192^2
// field, segments 2-7: {0, 1, 13, 14} kept in LDS for 54% of the symbols instead of {0, 1, 2, 4}
// for 86%). A table whose counts all sit at the floor keeps them.
static void context_shares(const uint8_t* host, uint64_t nf_off, double pi[kO1Ctx]) {
    double T[kO1Ctx][kO1Ctx] = {};
    for (int a = 0; a < kO1Ctx; a++) {
        for (int floor_out = 1; floor_out >= 0; floor_out--) {
            double tot = 0;
            for (int b = 0; b < kO1Ctx; b++) T[a][b] = 0;
            for (int sy = 0; sy < kO1Sym; sy++) {
                int16_t v;
                memcpy(&v, host + nf_off + 2 * ((size_t)a * kO1Sym + sy), 2);
                const double w = floor_out ? (v > 1 ? (double)v : 0.0) : (v == -1 ? 1.0 : (v > 0 ? (double)v : 0.0));
                if (w == 0) continue;
                tot += w;
                if (sy == 255) {
                    T[a][13] += w / 2;
                    T[a][14] += w / 2;
                } else {
                    T[a][o1_ctx((int)((sy >> 1) ^ (~(sy & 1) + 1)))] += w;
                }
            }
            if (tot > 0) {
                for (int b = 0; b < kO1Ctx; b++) T[a][b] /= tot;
                break;
            }
        }
    }
    for (int a = 0; a < kO1Ctx; a++) pi[a] = 1.0 / kO1Ctx;
    for (int it = 0; it < 64; it++) {
        double nx[kO1Ctx] = {};
        for (int a = 0; a < kO1Ctx; a++)
            for (int b = 0; b < kO1Ctx; b++) nx[b] += pi[a] * T[a][b];
        for (int b = 0; b < kO1Ctx; b++) pi[b] = nx[b];
    }
}

// The four consecutive contexts the walk keeps in LDS for a chain of the segment at nf_off: the
// window with the largest share (ties: the higher window, so 11..14 where escapes dominate).
static uint32_t hot_window(const double pi[kO1Ctx]) {
    uint32_t best = kWalkCtx0;
    double bw = -1;
    for (int h = kO1Ctx - kWalkCtxN; h >= 0; h--) {
        const double w = pi[h] + pi[h + 1] + pi[h + 2] + pi[h + 3];
        if (w > bw + 1e-12) { bw = w; best = (uint32_t)h; }
    }
    return best;
}

// The contexts of a segment's sequential chains that are kept in LDS: the largest by share, with both
// that follow an escape first where escapes are frequent (or where they are among the largest anyway).
static SerialMap serial_map(const double pi[kO1Ctx], double escapes, double bits) {
    int order[kO1Ctx];
    for (int a = 0; a < kO1Ctx; a++) order[a] = a;
    std::stable_sort(order, order + kO1Ctx, [&](int x, int y) { return pi[x] > pi[y]; });
    auto rank = [&](int c) { return (int)(std::find(order, order + kO1Ctx, c) - order); };
    SerialMap m{};
    m.esc = escapes > 1.0 / 64 || (rank(13) < kSerialHot && rank(14) < kSerialHot);
    if (m.esc)
        std::stable_sort(order, order + kO1Ctx, [&](int x, int y) {
            return (x >= 13 ? x - 13 : 2) < (y >= 13 ? y - 13 : 2);
        });
    for (int r = 0; r < kO1Ctx; r++) {
        m.inv_nibbles |= (uint64_t)r << (4 * order[r]);
        if (r < kSerialHot) m.perm_bytes |= (uint32_t)order[r] << (8 * r);
    }
    m.run = bits < kSerialRunBits ? kSerialRun : 0;
    return m;
}

// A chain as its call finds it, and how it is to be decoded.
struct O1Chain {
    O1Split k;
    SplitPlan plan;
    uint64_t seg;
    bool batched;  // handed to the batch
};

// The split chains of a call or of a batch, in launch order, and what their kernels left.
struct SplitRun {
    std::vector<O1Split> sc;
    std::vector<uint64_t> seg;
    O1SplitWs W{};
    unsigned int* stats = nullptr;
    uint64_t nlanes = 0, stream_bytes = 0, ncodes = 0;
    int cls_first[4];
    uint64_t cls_waves[3];
    size_t bytes = 0;  // device memory
    O1Split* dch = nullptr;
};
// 32-bit words of its statistics for nc chains: six counts, one a chain, then the pool's count.
static int split_stats(int nc) { return (6 + nc + 1) / 2 * 2 + 2; }

// Lays the chains out in the memory at `at`, those of one size class side by side for one launch each.
static void split_layout(const std::vector<O1Chain>& chains, SplitRun& R, uint8_t* at) {
    R = SplitRun{};
    std::vector<const O1Chain*> order;
    for (const O1Chain& c : chains) order.push_back(&c);
    std::stable_sort(order.begin(), order.end(), [](const O1Chain* x, const O1Chain* y) { return x->k.cls < y->k.cls; });
    uint64_t nparts = 0, ncand = 0, nwaves = 0;
    double pool = 0;
    std::fill(R.cls_first, R.cls_first + 4, 0);
    std::fill(R.cls_waves, R.cls_waves + 3, 0);
    for (const O1Chain* c : order) {
        R.sc.push_back(c->k);
        R.seg.push_back(c->seg);
        O1Split& k = R.sc.back();
        const uint64_t nw = split_waves(c->plan, k.nsub);
        k.tfirst = nparts;
        k.cfirst = ncand;
        k.wfirst = R.nlanes;
        k.gfirst = nwaves;
        nparts += k.nsub;
        ncand += (uint64_t)k.nsub * k.cap;
        R.nlanes += (((uint64_t)k.nsub << k.lgk) + 63) & ~63ull;
        nwaves += nw;
        R.cls_waves[k.cls] += nw;
        for (uint32_t z = k.cls + 1; z < 4; z++) R.cls_first[z] = (int)R.sc.size();
        pool += split_nodes(c->plan, k.m, k.nsub);
        R.stream_bytes += (uint64_t)k.len;
        R.ncodes += k.m;
    }
    const int nc = (int)R.sc.size();
    auto take = [&](auto*& p, uint64_t n) {
        p = reinterpret_cast<std::remove_reference_t<decltype(p)>>(at + R.bytes);
        R.bytes += (n * sizeof(*p) + 255) & ~(size_t)255;
    };
    O1SplitWs& W = R.W;
    W.nparts = nparts;
    W.pool_cap = std::min<uint64_t>((uint64_t)pool + 4096, kPoolMax);
    // FALCONS_O1_POOL_NODES: a test switch; the parts whose nodes find no room are decoded by the walk
    if (const char* few = getenv("FALCONS_O1_POOL_NODES")) W.pool_cap = std::min<uint64_t>(W.pool_cap, std::strtoull(few, nullptr, 10));
    take(R.dch, nc);
    take(W.cand, ncand);
    take(W.edge, ncand);
    take(W.exits, ncand);
    take(W.hdr, nparts * kSplitRounds);
    take(W.n0, nparts);
    take(W.wave, (nwaves + 1) * kSplitRounds);
    take(W.pool, W.pool_cap);
    take(W.res_state, nparts);
    take(W.res_e, nparts);
    take(W.res_off, nparts);
    const int nstats = split_stats(nc);
    take(R.stats, nstats);
    W.pool_used = reinterpret_cast<NodeCount*>(R.stats + nstats - 2);
}
// What split_layout takes beside its chains' split_bytes, at most: roundings, lists, a few nodes.
static size_t split_head(size_t nc) { return 65536 + (sizeof(O1Split) + 8) * nc; }
static void split_launch(const SplitRun& R, hipStream_t st) {
    const int nc = (int)R.sc.size(), nstats = split_stats(nc);
    const O1SplitWs& W = R.W;
    const int* cls_first = R.cls_first;
    O1Split* dch = R.dch;
    h2d(dch, R.sc.data(), R.sc.size(), st);
    FZ_HIP(hipMemsetAsync(R.stats, 0, nstats * sizeof(unsigned int), st));
    FZ_LAUNCH("o1_split_warm", 0, k_o1s_warm, dim3(nblk(R.nlanes)), dim3(256), 0, st, dch, nc, R.nlanes, W);
    for (int round = 0; round < kSplitRounds; round++)
        for (int z = 2; z >= 0; z--) {
            const int c0 = cls_first[z], cn = cls_first[z + 1] - c0;
            const uint32_t nw = (uint32_t)R.cls_waves[z];
            if (!cn || !nw) continue;
            if (z == kSplitFew)
                FZ_LAUNCH("o1_split_graph", 0, k_o1s_graph<kSplitNodes[0]>, dim3(nw), dim3(64), 0, st, dch + c0, cn, nw, round, W);
            else if (z == kSplitSome)
                FZ_LAUNCH("o1_split_graph", 0, k_o1s_graph<kSplitNodes[1]>, dim3(nw), dim3(64), 0, st, dch + c0, cn, nw, round, W);
            else
                FZ_LAUNCH("o1_split_graph", 0, k_o1s_graph<kSplitNodes[2]>, dim3(nw), dim3(64), 0, st, dch + c0, cn, nw, round, W);
        }
    FZ_LAUNCH("o1_split_walk", 0, k_o1s_walk, dim3(nc), dim3(kWalkThreads), 0, st, dch, nc, W, R.stats);
    FZ_LAUNCH("o1_split_out", R.stream_bytes + R.ncodes * 2, k_o1s_out, dim3(nblk(W.nparts)), dim3(256), 0, st, dch, nc, W);
    FZ_HIP(hipGetLastError());
}

// Sequential chains of several calls, decoded together (dense_batch_run).
struct DenseBatch {
    std::mutex mu;
    std::vector<SerialJob> jobs;
    std::vector<SerialTables> tabs;
    uint64_t bytes = 0, codes = 0;
    std::vector<O1Chain> split;
    double split_bytes = 0, split_limit = 0;
    SplitRun run;
};
DenseBatch* dense_batch_create() { return new DenseBatch; }
void dense_batch_destroy(DenseBatch* b) { delete b; }
size_t dense_batch_size(DenseBatch* b) {
    std::lock_guard<std::mutex> g(b->mu);
    return b->jobs.size() + b->split.size();
}
void dense_batch_limit(DenseBatch* b, size_t free_bytes) {
    std::lock_guard<std::mutex> g(b->mu);
    b->split_limit = std::min(kBatchSplitBytes, 0.25 * (double)free_bytes);
    // FALCONS_BATCH_SPLIT_BYTES: a test switch
    if (const char* most = getenv("FALCONS_BATCH_SPLIT_BYTES")) b->split_limit = std::min(b->split_limit, atof(most));
}
void dense_batch_clear(DenseBatch* b) {
    std::lock_guard<std::mutex> g(b->mu);
    b->jobs.clear();
    b->tabs.clear();
    b->bytes = b->codes = 0;
    b->split.clear();
    b->split_bytes = 0;
}
// Re-encodes the tables and decodes the chains of the lists on st; djobs and dtabs have room for them.
static void launch_serial(std::vector<SerialJob>& jobs, const std::vector<SerialTables>& tabs, SerialJob* djobs,
                          SerialTables* dtabs, uint64_t bytes, uint64_t codes, hipStream_t st) {
    FZ_LAUNCH("o1_serial_tables", 0, k_o1d_tables, dim3(kO1Ctx, (unsigned)tabs.size()), dim3(256), 0, st, dtabs);
    FZ_LAUNCH("o1_decode_serial", bytes + codes * 2, k_o1d_serial, dim3((unsigned)jobs.size()), dim3(kSerialThreads), 0, st,
              djobs);
    FZ_HIP(hipGetLastError());
}
// A stream waits for what was queued on the second one, however the block ends.
struct AuxJoin {
    const AuxStream& a;
    hipStream_t st;
    bool on;
    ~AuxJoin() {
        if (!on) return;
        (void)hipEventRecord(a.join, a.stream);
        (void)hipStreamWaitEvent(st, a.join, 0);
    }
};
void dense_batch_run(DenseBatch* b, DevArena& ws, hipStream_t st, const AuxStream& aux) {
    std::lock_guard<std::mutex> g(b->mu);
    const size_t n = b->jobs.size();
    if (n > 0x7fffffffu) throw std::length_error("too many sequential chains for one launch");
    if (b->tabs.size() > 65535u) throw std::length_error("too many sequential segments for one launch");
    // all device memory before the first launch: without it nothing of the batch is under way
    const size_t need = (size_t)b->split_bytes + split_head(b->split.size());
    uint8_t* mem = nullptr;
    if (!b->split.empty()) {
        mem = static_cast<uint8_t*>(ws.side(need, 0, (size_t)kBatchSplitBytes));
        if (!mem) throw GpuError("no device memory for the split chains of the batch");
    }
    SerialJob* dj = n ? ws.take<SerialJob>(n) : nullptr;
    SerialTables* dtab = n ? ws.take<SerialTables>(b->tabs.size()) : nullptr;
    // the two decoders beside each other (neither needs what the other writes); the sequential one, which
    // takes as long as its longest chain, is launched first
    const bool beside = n && mem && aux.stream;
    if (n) {
        // longest chains first, so that the last workgroups to start are short ones
        std::stable_sort(b->jobs.begin(), b->jobs.end(), [](const SerialJob& x, const SerialJob& y) { return x.m > y.m; });
        // the lists stay in b until dense_batch_clear, after the launches have finished
        h2d(dj, b->jobs.data(), n, st);
        h2d(dtab, b->tabs.data(), b->tabs.size(), st);
        if (beside) {
            FZ_HIP(hipEventRecord(aux.fork, st));
            FZ_HIP(hipStreamWaitEvent(aux.stream, aux.fork, 0));
        }
    }
    AuxJoin join{aux, st, beside};
    if (n) launch_serial(b->jobs, b->tabs, dj, dtab, b->bytes, b->codes, beside ? aux.stream : st);
    if (mem) {
        split_layout(b->split, b->run, mem);
        if (b->run.bytes > need) throw std::logic_error("split chains of the batch: more memory than planned");
        split_launch(b->run, st);
    }
}

// The lists of one call's chains. Copies on the call's stream read them: they stay until it has been waited for.
struct O1Lists {
    SplitRun split;
    std::vector<SerialJob> serial;
    std::vector<SerialTables> tabs;  // one a segment
};

// defer: the sequential chains are handed to it instead of launched, and the split ones that are short or
// find no room (their decode then runs in dense_batch_run, after the work this call has queued on st).
static void o1_decode_parallel(const uint8_t* host, const uint8_t* dev, const std::vector<uint64_t>& chains,
                               const std::vector<uint64_t>& nf_off, const DEntry* dt, const int16_t* ovf, int16_t* out,
                               int* err, DevArena& ws, hipStream_t st, const AuxStream& aux, DenseBatch* defer,
                               O1Lists& lists) {
    const int nch = (int)(chains.size() / 7);
    // FALCONS_O1_SEQUENTIAL=1 decodes every chain from its start; FALCONS_O1_PARALLEL_SHORT=1 splits
    // short chains too (the tests of either decoder on small fields)
    const char* seq_env = getenv("FALCONS_O1_SEQUENTIAL");
    const bool all_seq = seq_env && atoi(seq_env) != 0;
    const char* par_env = getenv("FALCONS_O1_PARALLEL_SHORT");
    const bool keep_short = par_env && atoi(par_env) != 0;
    // FALCONS_O1_GRAPH_NODES, FALCONS_O1_STAGE_NODES: test switches
    auto few_nodes = [](const char* v) { return v ? (uint32_t)std::strtoul(v, nullptr, 10) : ~0u; };
    const uint32_t graph_nodes = few_nodes(getenv("FALCONS_O1_GRAPH_NODES")), stage_nodes = few_nodes(getenv("FALCONS_O1_STAGE_NODES"));
    double pi[kO1Ctx];
    uint64_t pi_seg = ~0ull, ncodes = 0;
    std::vector<O1Chain> all;
    for (int q = 0; q < nch; q++) {
        const uint64_t* c = &chains[7 * q];
        const uint64_t m = c[3] - c[2];
        if (m == 0) continue;
        ncodes += m;
        // initial state: the tableLog bits under the end mark (FSE_initDState)
        const uint8_t* b = host + c[0];
        const int64_t top = (int64_t)(c[1] - 1) * 8 + (int64_t)highbit32(b[c[1] - 1]);
        uint32_t x0 = 0;
        for (int j = 1; j <= (int)kO1Log; j++) {
            const int64_t bit = top - j;
            x0 = (x0 << 1) | (bit >= 0 ? ((b[bit >> 3] >> (bit & 7)) & 1u) : 0u);
        }
        const int64_t pos0 = top - (int64_t)kO1Log;
        const double bits = (double)std::max<int64_t>(pos0, 0) / (double)m;
        if (pi_seg != c[5]) {
            context_shares(host, nf_off[c[5]], pi);
            pi_seg = c[5];
        }
        O1Chain x{};
        x.seg = c[5];
        x.batched = defer && m <= kDeferSymbols;
        SplitPlan& sp = x.plan;
        if (!all_seq) sp = split_plan(m, c[6], bits, pi, host + nf_off[c[5]], keep_short);
        if (x.batched && (sp.warm << sp.lgk) > kBatchWarm) {
            sp.lgk = 5;
            sp.warm = 1024;
        }
        O1Split& k = x.k;
        k.cb = dev + c[0];
        k.dt = reinterpret_cast<const uint32_t*>(dt + c[5] * kO1Ctx * (1u << kO1Log));
        k.ov = ovf + c[4];
        k.out = out + c[2];
        k.err = err;
        k.m = m;
        k.novf = c[6];
        k.len = (int64_t)c[1];
        k.pos0 = pos0;
        k.x0 = x0;
        if (sp.cls != kSplitNone) {
            k.sub_bits = split_sub_bits(sp, bits);
            k.nsub = (uint32_t)split_parts(pos0, k.sub_bits);
            k.warm_bits = (uint32_t)(bits * sp.warm) + 64;
            k.warm_steps = 2 * sp.warm;
            k.lgk = sp.lgk;
            k.cap = sp.cap;
            k.parts = sp.parts;
            k.max_sym = 8 * sp.sub;
            k.hot0 = hot_window(pi);
            k.cls = (uint32_t)sp.cls;
            k.max_nodes = std::min((uint32_t)kSplitNodes[sp.cls], graph_nodes);
            k.stage = std::min(walk_nodes((uint32_t)sp.cls), stage_nodes);
        }
        all.push_back(x);
    }
    // The split chains of this call, as many as its memory may hold; the others are decoded from their start. In a
    // batch, where the region of an item has no room for them, all of the item's go to the batch instead, which has
    // memory of its own.
    SplitRun& R = lists.split;
    {
        std::vector<SplitCand> cand;
        uint64_t serial = 0;
        double need = 0;
        for (O1Chain& x : all) {
            if (x.plan.cls == kSplitNone) serial = std::max(serial, x.k.m);
            else if (!x.batched) cand.push_back(SplitCand{&x.plan, x.k.m, x.k.nsub});
        }
        // what the call takes after this: the re-encoded tables of sequential chains, the scratch of a scan
        const size_t after = nf_off.size() * (sizeof(uint32_t) * kO1Ctx << kO1Log) + (1u << 20) + ncodes / 64;
        const double room = (double)std::min<uint64_t>(split_limit(ncodes), ws.side_room(after)) - 256.0 -
                            (double)split_head(cand.size());
        for (const SplitCand& x : cand) need += x.bytes();
        const bool to_batch = defer && need > room;
        if (!defer) split_choose(cand, room, serial);
        std::vector<O1Chain> own;
        need = (double)split_head(cand.size());
        for (O1Chain& x : all) {
            if (to_batch) x.batched = true;
            if (x.plan.cls == kSplitNone || x.batched) continue;
            need += split_bytes(x.plan, x.k.m, x.k.nsub);
            own.push_back(x);
        }
        if (!own.empty()) {
            if (uint8_t* mem = static_cast<uint8_t*>(ws.side((size_t)need, after, split_limit(ncodes)))) {
                split_layout(own, R, mem);
                if ((double)R.bytes > need) throw std::logic_error("split chains: more memory than planned");
            } else {
                for (O1Chain& x : all)
                    if (!x.batched) x.plan.cls = kSplitNone;
            }
        }
    }
    std::vector<SerialJob>& hd = lists.serial;
    std::vector<uint64_t> hd_seg;
    uint64_t dense_bytes = 0, dense_codes = 0;
    for (const O1Chain& x : all) {
        if (x.plan.cls != kSplitNone) {
            if (!x.batched) continue;
            const double need = split_bytes(x.plan, x.k.m, x.k.nsub);
            std::lock_guard<std::mutex> g(defer->mu);
            if (defer->split_bytes + need <= defer->split_limit) {
                defer->split.push_back(x);
                defer->split_bytes += need;
                continue;
            }
        }
        SerialJob k{};
        k.cb = x.k.cb;
        k.dt = x.k.dt;
        k.ov = x.k.ov;
        k.out = x.k.out;
        k.err = err;
        k.m = x.k.m;
        k.novf = x.k.novf;
        k.pos0 = x.k.pos0;
        k.x0 = x.k.x0;
        hd.push_back(k);
        hd_seg.push_back(x.seg);
        dense_bytes += (uint64_t)x.k.len;
        dense_codes += x.k.m;
    }
    // sequential chains run beside the rest, on the auxiliary stream when there is one
    hipStream_t dst = aux.stream ? aux.stream : st;
    const bool stats_on = getenv("FALCONS_DECODE_STATS") != nullptr;
    uint64_t* dense_times = nullptr;  // per sequential chain: clock at start and end (statistics only)
    std::vector<SerialTables>& tabs = lists.tabs;
    if (!hd.empty()) {
        for (size_t q = 0; q < hd.size();) {
            size_t q1 = q;
            double sm = 0, se = 0, sb = 0;
            for (; q1 < hd.size() && hd_seg[q1] == hd_seg[q]; q1++) {
                sm += (double)hd[q1].m;
                se += (double)hd[q1].novf;
                sb += (double)std::max<int64_t>(hd[q1].pos0, 0);
            }
            context_shares(host, nf_off[hd_seg[q]], pi);
            SerialTables t{hd[q].dt, ws.take<uint32_t>((size_t)kO1Ctx << kO1Log), serial_map(pi, se / sm, sb / sm)};
            for (; q < q1; q++) {
                hd[q].et = t.et;
                hd[q].map = t.map;
            }
            tabs.push_back(t);
        }
        if (stats_on && !defer) {
            dense_times = ws.take<uint64_t>(2 * hd.size());
            for (size_t q = 0; q < hd.size(); q++) hd[q].times = dense_times + 2 * q;
        }
    }
    if (!hd.empty() && defer) {
        std::lock_guard<std::mutex> g(defer->mu);
        defer->jobs.insert(defer->jobs.end(), hd.begin(), hd.end());
        defer->tabs.insert(defer->tabs.end(), tabs.begin(), tabs.end());
        defer->bytes += dense_bytes;
        defer->codes += dense_codes;
    } else if (!hd.empty()) {
        SerialJob* dj = ws.take<SerialJob>(hd.size());
        SerialTables* dtab = ws.take<SerialTables>(tabs.size());
        h2d(dj, hd.data(), hd.size(), st);
        h2d(dtab, tabs.data(), tabs.size(), st);
        // the second stream starts after every copy above
        if (aux.stream) {
            FZ_HIP(hipEventRecord(aux.fork, st));
            FZ_HIP(hipStreamWaitEvent(aux.stream, aux.fork, 0));
        }
        launch_serial(hd, tabs, dj, dtab, dense_bytes, dense_codes, dst);
    }
    AuxJoin join{aux, st, !hd.empty() && aux.stream != nullptr && !defer};
    if (R.sc.empty()) return;
    split_launch(R, st);
    const std::vector<O1Split>& sc = R.sc;
    const int nc = (int)sc.size();
    if (stats_on) {
        std::vector<unsigned int> hsv(split_stats(nc));
        d2h(hsv.data(), R.stats, hsv.size(), st);
        NodeCount nodes = 0;
        memcpy(&nodes, &hsv[hsv.size() - 2], sizeof(nodes));
        const unsigned int* hs = hsv.data();
        fprintf(stderr, "[o1 decode] chains (chain:exact subsequences/subsequences/escapes/bits a symbol/segment/"
                        "first LDS context of the walk/size class of its graphs):");
        for (int q = 0; q < nc; q++)
            fprintf(stderr, " %d:%u/%u/esc%llu/b%.2f/s%llu/h%u/c%u", q, hs[6 + q], sc[q].nsub, (unsigned long long)sc[q].novf,
                    (double)sc[q].pos0 / (double)std::max<uint64_t>(1, sc[q].m), (unsigned long long)R.seg[q],
                    sc[q].hot0, sc[q].cls);
        fprintf(stderr, "\n");
        fprintf(stderr, "[o1 decode] %zu chains decoded from their start:", hd.size());
        for (size_t q = 0; q < hd.size(); q++)
            fprintf(stderr, " b%.2f/s%llu/esc%llu", (double)hd[q].pos0 / (double)std::max<uint64_t>(1, hd[q].m),
                    (unsigned long long)hd_seg[q], (unsigned long long)hd[q].novf);
        fprintf(stderr, "\n");
        if (dense_times) {
            FZ_HIP(hipStreamSynchronize(dst));
            std::vector<uint64_t> tt(2 * hd.size());
            FZ_HIP(hipMemcpy(tt.data(), dense_times, tt.size() * sizeof(uint64_t), hipMemcpyDeviceToHost));
            fprintf(stderr, "[o1 decode] sequential chains (ms / ns a symbol / share of symbols in LDS contexts):");
            for (size_t q = 0; q < hd.size(); q++) {
                const double ms = (double)(tt[2 * q + 1] - tt[2 * q]) / 1e5;  // 100 MHz clock
                double ps[kO1Ctx];
                context_shares(host, nf_off[hd_seg[q]], ps);
                double share = 0;
                for (int r = 0; r < kSerialHot; r++) share += ps[hd[q].map.perm(r)];
                fprintf(stderr, " %.1f/%.0f/%.3f", ms, ms * 1e6 / (double)std::max<uint64_t>(1, hd[q].m), share);
            }
            fprintf(stderr, "\n");
        }
        fprintf(stderr, "[o1 decode] %d split chains, %llu parts, walk decoded %u exactly (%u without a whole path, %u "
                        "entries outside the set), %llu nodes of %llu\n",
                nc, (unsigned long long)R.W.nparts, hs[0] + hs[1], hs[0], hs[1], nodes, (unsigned long long)R.W.pool_cap);
    }
}

// Where the parts of an entropy stream sit (RleFseEncoder::save / encode, RleFse:897-982, 1072), read
// and checked on the host before anything runs on the device: every header, table, chain, escape
// stream and FSE block lies inside the stream, or the stream is refused as corrupt.
struct OvfPiece { uint64_t n, vcl_off, vman_off, nraw_off, mode, vbp, svcl; };
struct EntropyLayout {
    int method = 0, use_delta = 0;
    // method 1 (order-1 tANS)
    uint64_t S = 0, total_ovf = 0;
    std::vector<uint64_t> chains;  // 7 values a chain, see o1_decode_parallel
    std::vector<uint64_t> nf_off, ovf_base;
    std::vector<OvfPiece> pieces;
    // method 0 (RLE + FSE)
    uint64_t nr = 0, nv = 0, s_rcl = 0, s_vcl = 0, rbp = 0, vbp = 0, o_rcl = 0, o_vcl = 0, o_rman = 0, o_vman = 0;
};

static void parse_entropy(const uint8_t* host, size_t len, uint64_t n, EntropyLayout& Lay) {
    if (len < 5) throw std::invalid_argument("Truncated entropy stream");
    const uint8_t* const hend = host + len;
    auto need_in = [&](const uint8_t* at, uint64_t k) {
        if (at > hend || (uint64_t)(hend - at) < k) throw std::invalid_argument("Truncated entropy stream");
    };
    Lay.method = host[0] & 0x7F;
    Lay.use_delta = (host[0] & 0x80) != 0;
    if (Lay.method > 1) throw std::invalid_argument("corrupt entropy stream: unknown method");
    const uint8_t* hp = host + 5;
    if (Lay.method == 1) {
        need_in(hp, 8);
        uint64_t S = get64(hp);
        if (S > 16) throw std::invalid_argument("corrupt o1 tANS stream");
        if (!S) S = 1;
        const uint64_t seg = (n + S - 1) / S;
        Lay.S = S;
        std::vector<uint64_t>& chains = Lay.chains;
        std::vector<uint64_t>& nf_off = Lay.nf_off;
        std::vector<uint64_t>& ovf_base = Lay.ovf_base;
        std::vector<OvfPiece>& pieces = Lay.pieces;
        nf_off.assign(S, 0);
        ovf_base.assign(S, 0);
        pieces.assign(S, OvfPiece{});
        uint64_t total_ovf = 0;
        for (uint64_t g = 0; g < S; g++) {
            const uint64_t lo = g * seg, hi = std::min(lo + seg, n), sn = hi - lo;
            need_in(hp, 16);
            const uint64_t seg_n = get64(hp);
            const int K = (int)get64(hp);
            if (K < 1 || K > 16 || seg_n != sn) throw std::invalid_argument("corrupt o1 tANS stream");
            uint64_t blen[16], nvk[16];
            need_in(hp, 16 * (uint64_t)K);
            for (int k = 0; k < K; k++) blen[k] = get64(hp);
            for (int k = 0; k < K; k++) nvk[k] = get64(hp);
            nf_off[g] = (uint64_t)(hp - host);
            need_in(hp, kO1Ctx * kO1Sym * 2);
            hp += kO1Ctx * kO1Sym * 2;
            const uint64_t cs = sn ? (sn + K - 1) / K : 0;
            uint64_t ovfo = 0;
            for (int k = 0; k < K; k++) {
                const uint64_t clo = lo + k * cs, chi = std::min(clo + cs, hi);
                need_in(hp, blen[k]);
                if (chi > clo && (blen[k] == 0 || hp[blen[k] - 1] == 0)) throw std::invalid_argument("corrupt o1 tANS chain");
                if (nvk[k] > chi - std::min(chi, clo)) throw std::invalid_argument("corrupt o1 tANS escape count");
                chains.insert(chains.end(),
                              {(uint64_t)(hp - host), blen[k], clo, std::max(clo, chi), total_ovf + ovfo, g, nvk[k]});
                hp += blen[k];
                ovfo += nvk[k];
            }
            OvfPiece pc{ovfo, 0, 0, 0, 0, 0, 0};
            need_in(hp, 1);
            pc.mode = *hp++;
            if (ovfo) {
                if (pc.mode == 0) {
                    pc.nraw_off = (uint64_t)(hp - host);
                    need_in(hp, ovfo * 2);
                    hp += ovfo * 2;
                } else {
                    need_in(hp, 16);
                    const uint64_t svcl = get64(hp), vbp = get64(hp);
                    pc.vcl_off = (uint64_t)(hp - host);
                    need_in(hp, svcl);
                    hp += svcl;
                    pc.vman_off = (uint64_t)(hp - host);
                    pc.vbp = vbp;
                    pc.svcl = svcl;
                    std::vector<uint64_t> offs;
                    frame_offsets(host + pc.vcl_off, ovfo, svcl, offs);
                    need_in(hp, vbp);
                    if (vbp * 8 < ovfo) throw std::invalid_argument("corrupt o1 tANS escape stream");
                    hp += vbp;
                }
            }
            pieces[g] = pc;
            ovf_base[g] = total_ovf;
            total_ovf += ovfo;
        }
        Lay.total_ovf = total_ovf;
        return;
    }
    // [u64 nr, nv, s_rcl, s_vcl, rbp, vbp][fse_enc(rcl)][fse_enc(vcl)][rman][vman] (RleFse:972-979)
    need_in(hp, 48);
    const uint64_t nr = get64(hp), nv = get64(hp), s_rcl = get64(hp), s_vcl = get64(hp), rbp = get64(hp),
                   vbp = get64(hp);
    const uint64_t room = (uint64_t)(hend - hp);
    if (nr > n + 1 || nv > n || s_rcl > room || s_vcl > room - s_rcl || rbp > room - s_rcl - s_vcl ||
        vbp > room - s_rcl - s_vcl - rbp)
        throw std::invalid_argument("corrupt entropy stream: RLE header");
    const uint64_t o_rcl = (uint64_t)(hp - host), o_vcl = o_rcl + s_rcl, o_rman = o_vcl + s_vcl,
                   o_vman = o_rman + rbp;
    Lay.nr = nr; Lay.nv = nv; Lay.s_rcl = s_rcl; Lay.s_vcl = s_vcl; Lay.rbp = rbp; Lay.vbp = vbp;
    Lay.o_rcl = o_rcl; Lay.o_vcl = o_vcl; Lay.o_rman = o_rman; Lay.o_vman = o_vman;
    {
        std::vector<uint64_t> offs;
        frame_offsets(host + o_rcl, nr, s_rcl, offs);
        frame_offsets(host + o_vcl, nv, s_vcl, offs);
    }
}

void entropy_check(const uint8_t* host, size_t len, uint64_t n) {
    EntropyLayout Lay;
    parse_entropy(host, len, n, Lay);
}

// FSE blocks of several calls, decoded together (fse_batch_run): each call's blocks flag errors in
// the call's own flag.
struct FseBatch {
    std::mutex mu;
    std::vector<FseBlk> blks;  // pad: index into errs
    std::vector<int*> errs;
    bool big = false;  // a block takes the decoder's big layout
};
FseBatch* fse_batch_create() { return new FseBatch; }
void fse_batch_destroy(FseBatch* b) { delete b; }
void fse_batch_clear(FseBatch* b) {
    std::lock_guard<std::mutex> g(b->mu);
    b->blks.clear();
    b->errs.clear();
    b->big = false;
}

__global__ void k_or_flags(const int* src, int* const* dst, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && src[i]) *dst[i] = 1;
}

void fse_batch_run(FseBatch* b, DevArena& ws, hipStream_t st) {
    std::lock_guard<std::mutex> g(b->mu);
    if (b->blks.empty()) return;
    if (b->blks.size() > 0x7fffffffu) throw std::length_error("too many FSE blocks for one launch");
    const uint32_t ne = (uint32_t)b->errs.size();
    FseBlk* dblks = ws.take<FseBlk>(b->blks.size());
    int* gerr = ws.take<int>(ne);
    int** derr = ws.take<int*>(ne);
    // the lists stay in b until fse_batch_clear, after the launches have finished
    FZ_HIP(hipMemcpyAsync(dblks, b->blks.data(), b->blks.size() * sizeof(FseBlk), hipMemcpyHostToDevice, st));
    FZ_HIP(hipMemcpyAsync(derr, b->errs.data(), ne * sizeof(int*), hipMemcpyHostToDevice, st));
    FZ_HIP(hipMemsetAsync(gerr, 0, ne * sizeof(int), st));
    launch_fse_dec(b->big, dblks, b->blks.size(), gerr, st);
    FZ_LAUNCH("fse_dec_flags", 0, k_or_flags, dim3((ne + 255) / 256), dim3(256), 0, st, gerr, derr, ne);
    FZ_HIP(hipGetLastError());
}

// A decode in three parts (entropy_decode_start / middle / end); the state between them.
struct EntropyCall {
    EntropyLayout Lay;
    const uint8_t* host = nullptr;
    const uint8_t* dev = nullptr;
    uint64_t n = 0;
    int16_t* codes = nullptr;
    int16_t* out = nullptr;
    int* err = nullptr;
    int16_t* ovf = nullptr;       // method 1: escaped codes
    std::vector<uint8_t*> vcls;   // method 1: class bytes of every segment
    O1Lists lists;                // method 1: its chains; entropy_decode_end waits for what reads them
    uint8_t* rcl = nullptr;       // method 0: run and value classes
    uint8_t* vcl = nullptr;
};
EntropyCall* entropy_call_new() { return new EntropyCall; }
void entropy_call_free(EntropyCall* e) { delete e; }

void entropy_decode(const uint8_t* host, const uint8_t* dev, size_t len, uint64_t n, int16_t* codes, DevArena& ws,
                    hipStream_t st, const AuxStream& aux) {
    EntropyCall E;
    entropy_decode_start(&E, host, dev, len, n, codes, ws, st, nullptr);
    entropy_decode_middle(&E, ws, st, aux, nullptr);
    entropy_decode_end(&E, ws, st);
}

// Parses the stream and decodes its FSE-coded class bytes (escape classes of method 1, run and
// value classes of method 0), or hands their blocks to defer.
void entropy_decode_start(EntropyCall* E, const uint8_t* host, const uint8_t* dev, size_t len, uint64_t n,
                          int16_t* codes, DevArena& ws, hipStream_t st, FseBatch* defer) {
    parse_entropy(host, len, n, E->Lay);
    const EntropyLayout& Lay = E->Lay;
    E->host = host;
    E->dev = dev;
    E->n = n;
    E->codes = codes;
    E->err = ws.take<int>(1);
    FZ_HIP(hipMemsetAsync(E->err, 0, 4, st));
    E->out = Lay.use_delta ? ws.take<int16_t>(n + 1) : codes;
    std::vector<FseDecItem> fd;
    if (Lay.method == 1) {
        E->ovf = ws.take<int16_t>(Lay.total_ovf + 1);
        E->vcls.assign(Lay.S, nullptr);
        for (uint64_t g = 0; g < Lay.S; g++) {
            const OvfPiece& pc = Lay.pieces[g];
            if (!pc.n || pc.mode == 0) continue;
            E->vcls[g] = ws.take<uint8_t>(pc.n);
            fd.push_back(FseDecItem{host + pc.vcl_off, dev + pc.vcl_off, pc.n, pc.svcl, E->vcls[g]});
        }
    } else {
        E->rcl = ws.take<uint8_t>(Lay.nr + 1);
        E->vcl = ws.take<uint8_t>(Lay.nv + 1);
        fd = {{host + Lay.o_rcl, dev + Lay.o_rcl, Lay.nr, Lay.s_rcl, E->rcl},
              {host + Lay.o_vcl, dev + Lay.o_vcl, Lay.nv, Lay.s_vcl, E->vcl}};
    }
    if (!defer) {
        fse_dec_multi(fd, E->err, ws, st);
        return;
    }
    std::vector<FseBlk> blks;
    const bool big = fse_block_list(fd, blks);
    std::lock_guard<std::mutex> g(defer->mu);
    defer->big = defer->big || big;
    const uint32_t k = (uint32_t)defer->errs.size();
    defer->errs.push_back(E->err);
    for (FseBlk& b : blks) {
        b.pad = k;
        defer->blks.push_back(b);
    }
}

// Everything after the class bytes up to the decoded codes: method 1's escaped values, tables and
// chains (the sequential ones handed to defer when given), method 0's runs and values.
void entropy_decode_middle(EntropyCall* E, DevArena& ws, hipStream_t st, const AuxStream& aux, DenseBatch* defer) {
    const EntropyLayout& Lay = E->Lay;
    const uint8_t* host = E->host;
    const uint8_t* dev = E->dev;
    const uint64_t n = E->n;
    int* err = E->err;
    int16_t* out = E->out;
    if (Lay.method == 1) {
        const uint64_t S = Lay.S;
        const std::vector<uint64_t>& chains = Lay.chains;
        const std::vector<uint64_t>& nf_off = Lay.nf_off;
        const std::vector<uint64_t>& ovf_base = Lay.ovf_base;
        const std::vector<OvfPiece>& pieces = Lay.pieces;
        int16_t* ovf = E->ovf;
        for (uint64_t g = 0; g < S; g++) {
            const OvfPiece& pc = pieces[g];
            if (!pc.n) continue;
            if (pc.mode == 0) {
                FZ_HIP(hipMemcpyAsync(ovf + ovf_base[g], dev + pc.nraw_off, pc.n * 2, hipMemcpyDeviceToDevice, st));
            } else {
                uint8_t* vcl = E->vcls[g];
                uint64_t* voff = ws.take<uint64_t>(pc.n + 1);
                {
                    hipcub::TransformInputIterator<uint64_t, ToU64, const uint8_t*> it(vcl, ToU64{});
                    size_t b = 0;
                    FZ_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, b, it, voff, (int64_t)pc.n, st));
                    void* t = cub_scratch(ws, b);
                    FZ_HIP(hipcub::DeviceScan::ExclusiveSum(t, b, it, voff, (int64_t)pc.n, st));
                }
                FZ_LAUNCH("o1_escape_decode", pc.n * 3, k_ovf_values, dim3(nblk(pc.n)), dim3(256), 0, st, vcl, voff,
                          dev + pc.vman_off, pc.vbp * 8, pc.n, ovf + ovf_base[g], err);
                FZ_HIP(hipGetLastError());
            }
        }
        DEntry* dt = ws.take<DEntry>(S * kO1Ctx * (1u << kO1Log));
        uint64_t* dnf_off = ws.take<uint64_t>(S);
        h2d(dnf_off, nf_off.data(), S, st);
        FZ_LAUNCH("o1_dtables", 0, k_o1_dtables, dim3(kO1Ctx, (unsigned)S), dim3(256), 0, st, dev, dnf_off, dt, err);
        FZ_HIP(hipGetLastError());
        {  // the tables must be whole before any decoder reads them
            int herr = 0;
            d2h(&herr, err, 1, st);
            if (herr) throw std::invalid_argument("corrupt o1 tANS tables");
        }
        o1_decode_parallel(host, dev, chains, nf_off, dt, ovf, out, err, ws, st, aux, defer, E->lists);
    } else {
        const uint64_t nr = Lay.nr, nv = Lay.nv, rbp = Lay.rbp, vbp = Lay.vbp;
        const uint64_t o_rman = Lay.o_rman, o_vman = Lay.o_vman;
        uint8_t* rcl = E->rcl;
        uint8_t* vcl = E->vcl;
        // bit offsets of the mantissas
        uint64_t* rk = ws.take<uint64_t>(nr + 1);
        uint64_t* vk = ws.take<uint64_t>(nv + 1);
        uint64_t* roff = ws.take<uint64_t>(nr + 1);
        uint64_t* voff = ws.take<uint64_t>(nv + 1);
        {
            hipcub::TransformInputIterator<uint64_t, ToU64, const uint8_t*> ri(rcl, ToU64{});
            hipcub::TransformInputIterator<uint64_t, ToU64, const uint8_t*> vi(vcl, ToU64{});
            size_t b1 = 0, b2 = 0;
            FZ_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, b1, ri, roff, (int64_t)nr, st));
            void* t1 = cub_scratch(ws, b1);
            FZ_HIP(hipcub::DeviceScan::ExclusiveSum(t1, b1, ri, roff, (int64_t)nr, st));
            if (nv) {
                FZ_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, b2, vi, voff, (int64_t)nv, st));
                void* t2 = cub_scratch(ws, b2);
                FZ_HIP(hipcub::DeviceScan::ExclusiveSum(t2, b2, vi, voff, (int64_t)nv, st));
            }
        }
        (void)rk; (void)vk;
        uint64_t* runlen = ws.take<uint64_t>(nr + 1);
        uint64_t* runsum = ws.take<uint64_t>(nr + 1);
        FZ_LAUNCH("rle_runs_decode", 0, k_runs_decode, dim3(nblk(nr)), dim3(256), 0, st, rcl, roff, dev + o_rman, rbp * 8,
                  nr, runlen, err);
        FZ_HIP(hipGetLastError());
        {
            size_t b = 0;
            FZ_HIP(hipcub::DeviceScan::InclusiveSum(nullptr, b, runlen, runsum, (int64_t)nr, st));
            void* t = cub_scratch(ws, b);
            FZ_HIP(hipcub::DeviceScan::InclusiveSum(t, b, runlen, runsum, (int64_t)nr, st));
        }
        FZ_HIP(hipMemsetAsync(out, 0, n * 2, st));
        if (nv) FZ_LAUNCH("rle_values_place", 0, k_values_place, dim3(nblk(nv)), dim3(256), 0, st, vcl, voff, dev + o_vman,
                          vbp * 8, nv, runsum, n, out, err);
        FZ_HIP(hipGetLastError());
    }
}

void entropy_decode_end(EntropyCall* E, DevArena& ws, hipStream_t st) {
    if (E->Lay.use_delta && E->n > 0) {
        size_t b = 0;
        FZ_HIP(hipcub::DeviceScan::InclusiveScan(nullptr, b, E->out, E->codes, Add16{}, (int64_t)E->n, st));
        void* tmp = cub_scratch(ws, b);
        FZ_HIP(hipcub::DeviceScan::InclusiveScan(tmp, b, E->out, E->codes, Add16{}, (int64_t)E->n, st));
    }
    int herr = 0;
    d2h(&herr, E->err, 1, st);
    if (herr) throw std::runtime_error("corrupt entropy stream");
}
}  // namespace fz
