// Sort, scan and key-set steps of one 1024-thread block over at most 4096 keys
// in LDS: the whole of what a small batch's key sets need, in one launch
// instead of ten.
#pragma once
#include "engine.h"
#include "wave.h"

namespace cgd {

constexpr int kBsThreads = 1024, kBsWaves = kBsThreads / kWave;
constexpr int kBsItems = 4, kBsTile = kBsThreads * kBsItems;  // 4096 keys

struct BsLds {
    uint64_t key[kBsTile];
    uint32_t cnt[kBsWaves][256];
    uint32_t base[256];
    uint32_t sum[kBsWaves];
};

// Exclusive prefix of v over the block's threads; *total gets the sum.  L.sum
// may be reused after the caller's next __syncthreads.
__device__ __forceinline__ uint32_t BsScan(BsLds& L, uint32_t v, uint32_t* total) {
    const uint32_t w = threadIdx.x / kWave;
    const uint32_t incl = WaveInclusiveScan(v);
    if (LaneId() == kWave - 1) L.sum[w] = incl;
    __syncthreads();
    uint32_t pre = 0, tot = 0;
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)kBsWaves; i++) {
        const uint32_t s = L.sum[i];
        pre += i < w ? s : 0u;
        tot += s;
    }
    *total = tot;
    return pre + incl - v;
}

// Stable rank of a wave's keys by digit: `rounds` x 64 keys of the wave (k[r],
// valid[r]), earlier rounds first; pos[r] = keys of the wave with the same
// digit before this one; cnt (the wave's 256 counters, zeroed) ends at the
// wave's digit counts.  No block synchronisation: the counters are the wave's.
template <int kMax>
__device__ __forceinline__ void BsRank(uint32_t* cnt, uint32_t rounds, const uint64_t* k, uint32_t valid_mask,
                                       uint32_t shift, uint32_t* pos) {
#pragma unroll
    for (int r = 0; r < kMax; r++) {
        if ((uint32_t)r >= rounds) break;
        const bool valid = (valid_mask >> r) & 1u;
        const uint32_t d = (uint32_t)(k[r] >> shift) & 255u;
        uint64_t m = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; b++) {
            const uint64_t bb = __ballot((d >> b) & 1u);
            m &= ((d >> b) & 1u) ? bb : ~bb;
        }
        const uint32_t rank = RankBelow(m);
        const uint32_t prior = cnt[d];
        WaveSync();
        if (valid && rank == 0) cnt[d] = prior + (uint32_t)__popcll(m);
        WaveSync();
        pos[r] = prior + rank;
    }
}

// Sorts L.key[0..n) (n <= kBsTile) by the low `bits` bits; every thread calls.
// Up to 64 keys: one wavefront's bitonic network on registers; more: stable
// 8-bit digit passes, each wave ranking its own run of keys.
__device__ __forceinline__ void BlockSort(BsLds& L, uint32_t n, uint32_t bits) {
    const uint32_t t = threadIdx.x, w = t / kWave, lane = LaneId();
    __syncthreads();
    if (n <= (uint32_t)kWave) {
        if (w == 0) {
            uint64_t k = lane < n ? L.key[lane] : ~0ull;
#pragma unroll
            for (uint32_t size = 2; size <= 64; size <<= 1)
#pragma unroll
                for (uint32_t step = size >> 1; step > 0; step >>= 1) {
                    const uint64_t o = __shfl_xor((unsigned long long)k, (int)step, kWave);
                    const bool up = (lane & size) == 0, low = (lane & step) == 0;
                    const uint64_t lo = k < o ? k : o, hi = k < o ? o : k;
                    k = up == low ? lo : hi;
                }
            if (lane < n) L.key[lane] = k;
        }
        __syncthreads();
        return;
    }
    const uint32_t rounds = (n + kBsThreads - 1) / kBsThreads, per = rounds * kWave;
    for (uint32_t shift = 0; shift < bits; shift += 8) {
        for (uint32_t i = t; i < (uint32_t)kBsWaves * 256; i += kBsThreads) (&L.cnt[0][0])[i] = 0;
        uint64_t k[kBsItems];
        uint32_t pos[kBsItems], valid = 0;
#pragma unroll
        for (int r = 0; r < kBsItems; r++) {
            const uint32_t i = w * per + r * kWave + lane;
            const bool v = (uint32_t)r < rounds && i < n;
            k[r] = v ? L.key[i] : 0ull;
            valid |= v ? 1u << r : 0u;
        }
        __syncthreads();
        BsRank<kBsItems>(L.cnt[w], rounds, k, valid, shift, pos);
        __syncthreads();
        uint32_t all = 0;
        if (t < 256) {
            for (int i = 0; i < kBsWaves; i++) {
                const uint32_t c = L.cnt[i][t];
                L.cnt[i][t] = all;
                all += c;
            }
        }
        uint32_t total;
        const uint32_t ex = BsScan(L, all, &total);
        if (t < 256) L.base[t] = ex;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kBsItems; r++)
            if ((valid >> r) & 1u) {
                const uint32_t d = (uint32_t)(k[r] >> shift) & 255u;
                L.key[L.base[d] + L.cnt[w][d] + pos[r]] = k[r];
            }
        __syncthreads();
    }
}

}  // namespace cgd
