// Order-1 tANS decoder: which chains are split, and what that takes of device memory. Host rules without a
// kernel (fz_entropy.hip has the kernels), and the rule by which the graph waves share their pool.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#ifndef FZ_HD
#ifdef __HIPCC__
#define FZ_HD __host__ __device__ inline
#else
#define FZ_HD inline
#endif
#endif

namespace fz {

constexpr int kO1Ctx = 15;        // RleFseEncoder.hpp:344
constexpr int kO1Sym = 256;       // :347 (255 = escape to the side stream)
constexpr unsigned kO1Log = 13;   // :345

constexpr int kSplitRounds = 3;
constexpr uint32_t kSplitMaxCap = 128;  // candidates a part holds at most

// The nodes of all graph waves of a call go to one pool. Every wave of every round adds its number of
// nodes to one count, also when the pool is full, and 1,500 million codes with an escape in 20 make more
// than 2^32 of them (3 nodes a code): the count has 64 bits, so that a wave that finds the pool
// full keeps finding it full. First nodes are kept in 32 bits (all ones: no room).
typedef unsigned long long NodeCount;
constexpr uint32_t kPoolNone = ~0u;
constexpr uint64_t kPoolMax = 0xF0000000ull;
static_assert(kPoolMax < kPoolNone, "a first node is never taken for no room");

// Where a wave's nn nodes go when the count was `before`; kPoolNone: they do not fit.
FZ_HD uint32_t pool_first(NodeCount before, uint32_t nn, uint64_t cap) {
    return before + nn <= cap ? (uint32_t)before : kPoolNone;
}

// Chains of fewer symbols, or of fewer bits a symbol (where decoders started at guessed states hardly
// ever meet), are decoded from their start.
constexpr uint64_t kSplitMinSymbols = 8192;
constexpr double kSplitMinBits = 2.5;

// How a chain is decoded: from its start by one workgroup (k_o1d_serial), or split into parts. The
// split decoder follows, for every part, all states that its entry may be; what that costs is the
// number of such states that live side by side, estimated from the chain's tables:
//   mu   rate per symbol at which two decoders meet. It falls with the bits a symbol takes (a step
//        replaces that many bits of the 13-bit state): 5e-4 at 7.4 bits, 3e-4 at 6.2, 5e-5 at 3.2
//        (measured on k^-3 fields), so 8e-6 * 2^(0.85 bits).
//   pe   escapes per symbol by the tables, which is what a decoder off the true path meets. Every escape
//        doubles the paths and meeting halves them: about 1 + 2 pe / mu live ones
//        (counted on the CPU: 24 at 7.8 bits and an escape in 175 symbols, 130 at 7.4 and one in 36,
//        over 900 at 3.0 and one in 250).
// Where the lines between the two lie (ms split / from the start, limits off, cubes of float32; "spikes": a k^-3
// field with random values of 1,000 times the bound added):
//   from 6 bits on the nodes a symbol decide, 1.5 pe live: k^-3 200^3 at 5.9 of them 61 / 137, 64^3 at 8.7
//     3.3 / 5.4; at 17 to 25 133 / 133 and 10 / 5.6. The line stands at 6, where parts begin to outgrow
//     the largest table (1,024 nodes a round).
//   4.5 to 6 bits, spikes 160^3: 23 to 34 live 16 / 114, 68 to 100 12 / 115, 215 to 319 198 / 120. The line is 60.
//   below, spikes 160^3: 4 to 5 live 4.6 / 109, 13 to 19 30 / 110, 37 to 55 18 / 112, 110 to 165 30 / 111, 344 to 518
//     210 / 123. The line is 10.
// Both lower lines stand well in front of where the two decoders cost the same.
// Split chains, by size class of the graph kernel; kSplitNone: from the start.
enum { kSplitFew = 0, kSplitSome = 1, kSplitMany = 2, kSplitNone = 3 };
constexpr int kSplitNodes[3] = {128, 512, 1024};
struct SplitPlan {
    int cls = kSplitNone;
    double nodes = 0;  // nodes a symbol
    double room = 0;   // nodes a symbol that the pool has room for
    uint32_t lgk = 0, warm = 0, cap = 0, parts = 0, sub = 0;  // warm, sub in symbols
};
// m symbols, novf escapes, pi: shares of the contexts, norm: the segment's normalized counts (int16).
inline SplitPlan split_plan(uint64_t m, uint64_t novf, double bits, const double pi[kO1Ctx], const uint8_t* norm,
                            bool keep_short) {
    SplitPlan s;
    // a chain of few symbols is done sooner from its start than the split decoder's launches take
    if (m < (keep_short ? 4096u : kSplitMinSymbols) || bits < kSplitMinBits) return s;
    double pe = 0;
    for (int a = 0; a < kO1Ctx; a++) {
        int16_t v;
        memcpy(&v, norm + 2 * ((size_t)a * kO1Sym + 255), 2);
        pe += pi[a] * (v < 0 ? 1.0 : (double)v) / (double)(1u << kO1Log);
    }
    // the first chain of a segment holds most of its escapes (the coarse levels)
    pe = std::max(pe, 0.25 * (double)novf / (double)m);
    const double mu = 8e-6 * std::exp2(0.85 * bits);
    const double live = 1.0 + 2.0 * pe / mu;
    if (novf * 8 > m || live > (bits >= 6.0 ? 200.0 : bits >= 4.5 ? 60.0 : 10.0)) return s;
    s.nodes = 1.5 * pe * live;
    // Nodes counted over the three rounds for one of the estimate, k^-3 fields, spikes, fronts and integers: 0.6 to
    // 0.9 from 6.5 bits on, up to 1.2 below.
    s.room = (bits >= 6.5 ? 1.0 : 1.4) * s.nodes;
    if (pe < 1.0 / 1024 && live <= 10.0) {
        // Few states: long parts, and guessed decoders enough, early enough, for the true entry to be
        // among their states in most parts before the first round (CPU counts on k^-3 fields, parts
        // that the walk decodes exactly after three rounds: 6.2 bits, 8 decoders 512 symbols ahead 1 of
        // 2000; 3.2 bits, 64 decoders 2048 ahead 2 of 750, 32 decoders 7).
        s.cls = kSplitFew;
        s.sub = m >= (1u << 20) ? (bits >= 5.5 ? 1024 : 2048) : m >= (1u << 18) ? 1024 : m >= (1u << 16) ? 512 : 256;
        s.warm = bits >= 5.5 ? 512 : 2048;
        s.lgk = bits >= 6.0 ? 3 : bits >= 5.5 ? 4 : 6;
        s.cap = s.lgk <= 4 ? 16 : 32;
        s.parts = s.lgk <= 4 ? 16 : 8;
        while (s.parts > 1 && s.parts * s.nodes * s.sub > kSplitNodes[kSplitFew] / 3) s.parts /= 2;
    } else {
        // Escapes saturate the sets in a round or two whatever they start from: short parts and a short
        // warm-up (same counts: none of 500 parts left at 16 decoders 256 symbols ahead).
        s.sub = 256;
        s.warm = 256;
        s.lgk = 4;
        const double nodes = s.nodes * s.sub;
        // past its table a graph is lost to the walk
        if (nodes > 1.5 * kSplitNodes[kSplitMany]) return s;
        s.cls = nodes <= kSplitNodes[kSplitSome] / 4 ? kSplitSome : kSplitMany;
        s.cap = s.cls == kSplitSome ? 64 : kSplitMaxCap;
        s.parts = s.cls == kSplitMany ? 1 : nodes <= kSplitNodes[kSplitSome] / 16 ? 4 : nodes <= kSplitNodes[kSplitSome] / 8 ? 2 : 1;
    }
    return s;
}

// Parts of a chain that ends at read position pos0, and the bits of one.
inline uint32_t split_sub_bits(const SplitPlan& s, double bits) { return (uint32_t)std::max(2048.0, bits * s.sub); }
inline uint64_t split_parts(int64_t pos0, uint32_t sub_bits) {
    return (uint64_t)std::max<int64_t>(1, (pos0 + sub_bits - 1) / sub_bits);
}
inline uint64_t split_waves(const SplitPlan& s, uint64_t nsub) { return (nsub - 1 + s.parts - 1) / s.parts; }

// Nodes of the pool that are a chain's share: what the plan makes room for, and some for each wave, which
// small graphs live on. (The pool held four times the estimate, 18.6 nodes a code where 3 were used, 14.8 GB for a
// 512^3 field at REL 3.3e-4; a chain past its share is decoded all the same, the parts without room by the walk.)
inline double split_nodes(const SplitPlan& s, uint64_t m, uint64_t nsub) {
    return s.room * (double)m + (s.cls == kSplitFew ? 64.0 : 32.0) * (double)split_waves(s, nsub);
}
// Device bytes of a chain: sets, words a part, words a wave, nodes.
inline double split_bytes(const SplitPlan& s, uint64_t m, uint64_t nsub) {
    return (12.0 * s.cap + 27.0) * (double)nsub + 8.0 * kSplitRounds * (double)split_waves(s, nsub) +
           8.0 * split_nodes(s, m, nsub);
}

// Most device bytes that the split chains of a call of n codes take; callers that admit calls by their
// workspace count them beside what every call takes. 64 a code hold nearly every plan of a field of one segment
// (16.8 million codes), where splitting saves most (a quarter of the field is one chain: 256^3 at REL 5e-4
// 64 ms, 289 from the start). Fields of many segments have short chains and few segments with many
// escapes: 512^3 takes 3 bytes a code at REL 8e-4 (44 ms, 204 from the start).
inline uint64_t split_limit(uint64_t n) { return std::min<uint64_t>(64 * n, (1ull << 30) + 4 * n); }

// Nodes of all split chains, for one symbol of the longest chain that is decoded from its start, above which splitting
// the others does not pay: the call takes as long as that chain (66 ns a symbol) anyhow, and the graphs beside
// it slow it (1 ns a node). Measured, ms with and without the others split: 512^3 at REL 7e-4, 7 nodes, 155 / 162; at
// 4e-4, 11 nodes, 153 / 170; 384^3 at 3.6e-4, 70 nodes, 167 / 161; 512^3 at 3.6e-4, 170 nodes, 204 / 166.
constexpr double kSplitMixed = 32.0;

// Takes chains out of the split ones (cls becomes kSplitNone) until what is left fits in `limit` bytes and
// pays: by bytes a symbol, the most first. serial: symbols of the longest chain of the call that is
// decoded from its start already, 0 for none.
struct SplitCand {
    SplitPlan* plan;
    uint64_t m, nsub;
    double bytes() const { return split_bytes(*plan, m, nsub); }
    double nodes() const { return plan->nodes * (double)m; }
};
inline void split_choose(std::vector<SplitCand>& c, double limit, uint64_t serial) {
    double total = 0, nodes = 0;
    for (const SplitCand& x : c) {
        total += x.bytes();
        nodes += x.nodes();
    }
    std::stable_sort(c.begin(), c.end(), [](const SplitCand& x, const SplitCand& y) {
        return x.bytes() * (double)y.m > y.bytes() * (double)x.m;
    });
    for (SplitCand& x : c) {
        if (total <= limit && !(serial && nodes > kSplitMixed * (double)serial)) return;
        total -= x.bytes();
        nodes -= x.nodes();
        x.plan->cls = kSplitNone;
        serial = std::max(serial, x.m);
    }
}

}  // namespace fz
