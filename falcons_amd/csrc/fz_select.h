// Order-preserving selection of the codes that a test holds for (stream compaction): one workgroup
// per tile counts its hits, a scan of the tile counts gives each tile its output offset, and a second
// pass hands out the hits of every tile that has any, in index order. Tiles without hits are read once.
//
// A thread holds 16 consecutive codes (two 16-byte loads), a workgroup a tile of 4,096: the passes are
// bound by the read of the codes (2 bytes each) for long arrays, and by the number of workgroups in
// flight for short ones. Tiles of 65,536 codes read two bytes a thread at a time left a chunk of
// 540,000 codes on 9 of 256 CUs. Count, scan, hand-out and what gathered the values, on those tiles and here, escapes
// of order-1 coding: 0.16 -> 0.02 ms (86,000 codes), 0.32 -> 0.08 ms (134 million, one code in 2,700 an escape),
// 0.74 -> 0.29 ms (134 million, one in two); a batch of 192 chunks of 540,000 codes decodes in 64 ms where it took 76.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "fz_common.h"

namespace fz {

constexpr uint32_t kSelLane = 16;                // codes of a thread
constexpr uint64_t kSelTile = 256 * kSelLane;

// Bit k: test holds for codes[i0 + k] (bits at and past n are 0).
template <class Test>
__device__ __forceinline__ uint32_t sel_mask(const int16_t* codes, uint64_t i0, uint64_t n, Test test) {
    uint32_t m = 0;
    if (i0 + kSelLane <= n && ((uintptr_t)codes & 15u) == 0) {
        const uint4* p = reinterpret_cast<const uint4*>(codes + i0);
        const uint4 a = p[0], b = p[1];
        const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int r = 0; r < 8; r++) {
            m |= (test((int16_t)w[r]) ? 1u : 0u) << (2 * r);
            m |= (test((int16_t)(w[r] >> 16)) ? 1u : 0u) << (2 * r + 1);
        }
    } else if (i0 < n) {
        for (uint32_t k = 0; k < kSelLane && i0 + k < n; k++) m |= (test(codes[i0 + k]) ? 1u : 0u) << k;
    }
    return m;
}

template <class Test>
__global__ void __launch_bounds__(256) k_sel_count(const int16_t* codes, uint64_t n, Test test, uint32_t* counts) {
    __shared__ uint32_t part[4];
    const uint64_t i0 = (uint64_t)blockIdx.x * kSelTile + threadIdx.x * kSelLane;
    uint32_t c = __popc(sel_mask(codes, i0, n, test));
#pragma unroll
    for (int d = 32; d; d >>= 1) c += __shfl_xor(c, d, 64);
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// offs[t] = hits in the tiles before t, *total = all hits. One workgroup: 4,096 tiles a round (16
// million codes), so that a launch is all that most arrays pay.
static __global__ void __launch_bounds__(1024) k_sel_scan(const uint32_t* counts, uint64_t ntiles, uint64_t* offs,
                                                          uint64_t* total) {
    __shared__ uint32_t part[16];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint64_t base = 0;
    for (uint64_t t0 = 0; t0 < ntiles; t0 += 4096) {
        const uint64_t t = t0 + 4 * threadIdx.x;
        uint32_t c[4];
#pragma unroll
        for (int k = 0; k < 4; k++) c[k] = t + k < ntiles ? counts[t + k] : 0u;
        const uint32_t own = c[0] + c[1] + c[2] + c[3];  // sums of up to 2^17 a tile fit
        uint32_t inc = own;
#pragma unroll
        for (uint32_t d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(inc, d, 64);
            if (lane >= d) inc += y;
        }
        if (lane == 63) part[wave] = inc;
        __syncthreads();
        uint32_t before = 0, all = 0;
#pragma unroll
        for (uint32_t w = 0; w < 16; w++) {
            const uint32_t v = part[w];
            before += w < wave ? v : 0u;
            all += v;
        }
        __syncthreads();
        uint64_t o = base + before + inc - own;
#pragma unroll
        for (int k = 0; k < 4; k++) {
            if (t + k < ntiles) offs[t + k] = o;
            o += c[k];
        }
        base += all;
    }
    if (threadIdx.x == 0) *total = base;
}

// emit(k, i): the k-th hit is code i.
template <class Test, class Emit>
__global__ void __launch_bounds__(256) k_sel_write(const int16_t* codes, uint64_t n, Test test, const uint32_t* counts,
                                                   const uint64_t* offs, Emit emit) {
    __shared__ uint32_t part[4];
    const uint64_t t = blockIdx.x;
    if (counts[t] == 0) return;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t i0 = t * kSelTile + threadIdx.x * kSelLane;
    uint32_t m = sel_mask(codes, i0, n, test);
    const uint32_t own = __popc(m);
    uint32_t inc = own;
#pragma unroll
    for (uint32_t d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(inc, d, 64);
        if (lane >= d) inc += y;
    }
    if (lane == 63) part[wave] = inc;
    __syncthreads();
    uint64_t k = offs[t] + inc - own;
    for (uint32_t w = 0; w < wave; w++) k += part[w];
    for (; m; m &= m - 1) emit(k++, i0 + __ffs(m) - 1);
}

// below[q] = hits under ends[q] (at most n), from the tiles' offsets and the codes of one tile; one
// workgroup an end.
template <class Test>
__global__ void __launch_bounds__(256) k_sel_below(const int16_t* codes, uint64_t n, Test test, const uint64_t* offs,
                                                   uint64_t ntiles, const uint64_t* total, const uint64_t* ends,
                                                   uint64_t* below) {
    __shared__ uint32_t part[4];
    const uint64_t end = min(ends[blockIdx.x], n), t = end / kSelTile;
    const uint64_t i0 = t * kSelTile + threadIdx.x * kSelLane;
    uint32_t c = i0 < end ? __popc(sel_mask(codes, i0, end, test)) : 0u;
#pragma unroll
    for (int d = 32; d; d >>= 1) c += __shfl_xor(c, d, 64);
    if ((threadIdx.x & 63u) == 0) part[threadIdx.x >> 6] = c;
    __syncthreads();
    if (threadIdx.x == 0)
        below[blockIdx.x] = (t < ntiles ? offs[t] : *total) + part[0] + part[1] + part[2] + part[3];
}

// Tile counts and offsets of a selection over n codes, in scratch of select_scratch_bytes(n).
struct SelTiles {
    uint64_t n, count;
    uint64_t* offs;
    uint32_t* counts;
    SelTiles(void* scratch, uint64_t n_)
        : n(n_), count((n_ + kSelTile - 1) / kSelTile), offs(static_cast<uint64_t*>(scratch)),
          counts(reinterpret_cast<uint32_t*>(offs + count)) {}
};
inline size_t select_scratch_bytes(uint64_t n) { return ((n + kSelTile - 1) / kSelTile) * 12 + 16; }

// Hands every hit to emit, ascending; *total_dev = their number.
template <class Test, class Emit>
SelTiles select_codes(const int16_t* codes, uint64_t n, Test test, Emit emit, uint64_t* total_dev, void* scratch,
                      const char* name, hipStream_t st) {
    const SelTiles T(scratch, n);
    ProfScope ps(name, n * 2, st);
    const unsigned nt = (unsigned)T.count;
    if (nt) hipLaunchKernelGGL(k_sel_count<Test>, dim3(nt), dim3(256), 0, st, codes, n, test, T.counts);
    hipLaunchKernelGGL(k_sel_scan, dim3(1), dim3(1024), 0, st, T.counts, T.count, T.offs, total_dev);
    if (nt)
        hipLaunchKernelGGL((k_sel_write<Test, Emit>), dim3(nt), dim3(256), 0, st, codes, n, test, T.counts, T.offs, emit);
    FZ_HIP(hipGetLastError());
    return T;
}

struct SelIndex {
    uint64_t* out;
    __device__ __forceinline__ void operator()(uint64_t k, uint64_t i) const { out[k] = i; }
};
// out[0 .. *total_dev) = the indices i < n whose code the test holds for, ascending.
template <class Test>
void select_indices(const int16_t* codes, uint64_t n, Test test, uint64_t* out, uint64_t* total_dev, void* scratch,
                    const char* name, hipStream_t st) {
    (void)select_codes(codes, n, test, SelIndex{out}, total_dev, scratch, name, st);
}

// The quantizer's escape code.
struct IsEscape {
    __device__ __forceinline__ bool operator()(int16_t c) const { return c == -32768; }
};

}  // namespace fz
