// Device-wide primitives for gfx950: exclusive scan (reduce-then-scan) and a
// stable LSD radix sort of u64 keys with 8-bit digits.  These replace the
// thrust::sort / unique and CUB scan calls of the reference
// (index/calig_helper_gamma.cu:304, 491-492, 573; graph/graph_gpu.cu:1395-1400).
#include <atomic>
#include <chrono>
#include <cstring>

#include "blocksort.h"
#include "engine.h"
#include "wave.h"

namespace cgd {

namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;  // 2048

template <class T>
__device__ T BlockExclusiveScan(T v, T* total) {
    __shared__ T wsum[kScanThreads / kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    T inc = WaveInclusiveScan(v);
    if (lane == kWave - 1) wsum[w] = inc;
    __syncthreads();
    T pre = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < kScanThreads / kWave; i++) {
        if (i < w) pre += wsum[i];
        tot += wsum[i];
    }
    __syncthreads();
    *total = tot;
    return pre + inc - v;
}

template <class T>
__global__ void __launch_bounds__(kScanThreads) KScanReduce(const T* in, uint64_t n, T* tile_sums) {
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
    T s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        uint64_t idx = base + (uint64_t)threadIdx.x * kScanItems + i;
        if (idx < n) s += in[idx];
    }
    T tot;
    BlockExclusiveScan(s, &tot);
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = tot;
}

// Single block scans the tile sums in place and writes the grand total.
template <class T>
__global__ void __launch_bounds__(kScanThreads) KScanTiles(T* tile_sums, uint64_t nt, uint64_t* total) {
    T carry = 0;
    for (uint64_t base = 0; base < nt; base += kScanThreads) {
        uint64_t idx = base + threadIdx.x;
        T v = idx < nt ? tile_sums[idx] : 0;
        T tot;
        T ex = BlockExclusiveScan(v, &tot);
        if (idx < nt) tile_sums[idx] = carry + ex;
        carry += tot;
    }
    if (threadIdx.x == 0 && total) *total = (uint64_t)carry;
}

template <class T>
__global__ void __launch_bounds__(kScanThreads) KScanApply(const T* in, T* out, uint64_t n, const T* tile_sums) {
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
    T v[kScanItems];
    T s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        uint64_t idx = base + i;
        v[i] = idx < n ? in[idx] : 0;
        s += v[i];
    }
    T tot;
    T ex = BlockExclusiveScan(s, &tot) + tile_sums[blockIdx.x];
#pragma unroll
    for (int i = 0; i < kScanItems; i++) {
        uint64_t idx = base + i;
        if (idx < n) out[idx] = ex;
        ex += v[i];
    }
}

// Whole scan in one block, tile after tile with a running carry (in place
// allowed: a tile is read into registers before it is written).  For short
// inputs one launch instead of three: the per-batch index kernels run dozens
// of such scans per query.
template <class T>
__global__ void __launch_bounds__(kScanThreads) KScanSingle(const T* in, T* out, uint64_t n, uint64_t* total) {
    T carry = 0;
    for (uint64_t base = 0; base < n; base += kScanTile) {
        const uint64_t b0 = base + (uint64_t)threadIdx.x * kScanItems;
        T v[kScanItems];
        T sum = 0;
#pragma unroll
        for (int i = 0; i < kScanItems; i++) {
            v[i] = b0 + i < n ? in[b0 + i] : 0;
            sum += v[i];
        }
        T tot;
        T ex = BlockExclusiveScan(sum, &tot) + carry;
#pragma unroll
        for (int i = 0; i < kScanItems; i++) {
            if (b0 + i < n) out[b0 + i] = ex;
            ex += v[i];
        }
        carry += tot;
    }
    if (threadIdx.x == 0 && total) *total = (uint64_t)carry;
}

constexpr uint64_t kScanSingleMax = 4 * kScanTile;  // 8192 elements (the block walks its tiles in turn)

template <class T>
void ScanImpl(const T* in, T* out, uint64_t n, uint64_t* total_dev, void* scratch, hipStream_t s) {
    if (n == 0) {
        if (total_dev) FillU64(total_dev, 0, 1, s);
        return;
    }
    if (n <= kScanSingleMax) {
        KScanSingle<T><<<1, kScanThreads, 0, s>>>(in, out, n, total_dev);
        CGD_HIP(hipGetLastError());
        return;
    }
    const uint64_t nt = (n + kScanTile - 1) / kScanTile;
    T* tiles = (T*)scratch;
    KScanReduce<T><<<(unsigned)nt, kScanThreads, 0, s>>>(in, n, tiles);
    KScanTiles<T><<<1, kScanThreads, 0, s>>>(tiles, nt, total_dev);
    KScanApply<T><<<(unsigned)nt, kScanThreads, 0, s>>>(in, out, n, tiles);
    CGD_HIP(hipGetLastError());
}

__global__ void KFill64(uint64_t* p, uint64_t v, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}
__global__ void KSetWords(uint64_t* base, WordSet ws) {
    if (threadIdx.x < ws.n) base[ws.off[threadIdx.x]] = ws.val[threadIdx.x];
}
__global__ void KFill32(uint32_t* p, uint32_t v, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

// Words of a device block, then the sequence number, into coherent host memory.
__global__ void __launch_bounds__(256) KPublish(const uint64_t* __restrict__ src, uint32_t words, uint64_t* dst,
                                                uint64_t* seq_at, uint64_t seq) {
    for (uint32_t i = threadIdx.x; i < words; i += blockDim.x)
        __hip_atomic_store(&dst[i], src[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_store(seq_at, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// ---------------------------------------------------------------- radix sort
constexpr int kRsTile = kBsTile;  // keys per block

__global__ void __launch_bounds__(kBsThreads) KRsHist(const uint64_t* keys, uint64_t n, uint32_t shift,
                                                       uint32_t* hist, uint32_t nblocks) {
    __shared__ uint32_t h[256];
    if (threadIdx.x < 256) h[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * kRsTile;
#pragma unroll
    for (int i = 0; i < kBsItems; i++) {
        uint64_t idx = base + (uint64_t)i * kBsThreads + threadIdx.x;
        if (idx < n) atomicAdd(&h[(keys[idx] >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 256) hist[(uint64_t)threadIdx.x * nblocks + blockIdx.x] = h[threadIdx.x];
}

// Stable scatter of one tile: each wave ranks its own run of 256 keys among
// equal digits (BsRank, no block synchronisation between its rounds), the
// waves' digit counts give the rank across them.  With 256 threads and a block
// round of 256 keys (four barriers each) a tile took 14 us, this takes 5.
__global__ void __launch_bounds__(kBsThreads) KRsScatter(const uint64_t* in, uint64_t* out, uint64_t n,
                                                          uint32_t shift, const uint32_t* offs, uint32_t nblocks) {
    __shared__ uint32_t cnt[kBsWaves][256];
    const uint32_t t = threadIdx.x, w = t / kWave, lane = LaneId();
    const uint64_t base = (uint64_t)blockIdx.x * kRsTile;
    uint64_t k[kBsItems];
    uint32_t pos[kBsItems], valid = 0;
#pragma unroll
    for (int r = 0; r < kBsItems; r++) {
        const uint64_t i = base + w * (kBsItems * kWave) + r * kWave + lane;
        k[r] = i < n ? in[i] : 0ull;
        valid |= i < n ? 1u << r : 0u;
    }
    for (uint32_t i = t; i < (uint32_t)kBsWaves * 256; i += kBsThreads) (&cnt[0][0])[i] = 0;
    __syncthreads();
    BsRank<kBsItems>(cnt[w], kBsItems, k, valid, shift, pos);
    __syncthreads();
    if (t < 256) {
        uint32_t all = offs[(uint64_t)t * nblocks + blockIdx.x];
        for (int i = 0; i < kBsWaves; i++) {
            const uint32_t c = cnt[i][t];
            cnt[i][t] = all;
            all += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kBsItems; r++)
        if ((valid >> r) & 1u) out[cnt[w][(uint32_t)(k[r] >> shift) & 255u] + pos[r]] = k[r];
}

// Whole sort of at most one tile in one block.
__global__ void __launch_bounds__(kBsThreads) KRsSortTile(uint64_t* keys, uint32_t n, uint32_t bits) {
    __shared__ BsLds L;
    for (uint32_t i = threadIdx.x; i < n; i += kBsThreads) L.key[i] = keys[i];
    BlockSort(L, n, bits);
    for (uint32_t i = threadIdx.x; i < n; i += kBsThreads) keys[i] = L.key[i];
}

}  // namespace

size_t ScanScratchBytes(uint64_t n) { return ((n + kScanTile - 1) / kScanTile + 1) * sizeof(uint64_t); }

void ScanU32(const uint32_t* in, uint32_t* out, uint64_t n, uint64_t* total_dev, void* scratch, hipStream_t s) {
    ScanImpl<uint32_t>(in, out, n, total_dev, scratch, s);
}
void ScanU64(const uint64_t* in, uint64_t* out, uint64_t n, uint64_t* total_dev, void* scratch, hipStream_t s) {
    ScanImpl<uint64_t>(in, out, n, total_dev, scratch, s);
}

void FillU64(uint64_t* p, uint64_t v, uint64_t n, hipStream_t s) {
    if (!n) return;
    unsigned g = (unsigned)std::min<uint64_t>((n + 255) / 256, 4096);
    KFill64<<<g, 256, 0, s>>>(p, v, n);
}
void SetWords(uint64_t* base, const WordSet& ws, hipStream_t s) {
    if (ws.n) KSetWords<<<1, 64, 0, s>>>(base, ws);
}
void FillU32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t s) {
    if (!n) return;
    unsigned g = (unsigned)std::min<uint64_t>((n + 255) / 256, 4096);
    KFill32<<<g, 256, 0, s>>>(p, v, n);
}

void Mailbox::Alloc(size_t bytes) {
    void *h = nullptr, *d = nullptr;
    const size_t n = kHeader * 8 + bytes;
    CGD_HIP(hipHostMalloc(&h, n, hipHostMallocMapped | hipHostMallocCoherent));
    host_ = (uint64_t*)h;
    memset(h, 0, n);
    CGD_HIP(hipHostGetDevicePointer(&d, h, 0));
    dev_ = (uint64_t*)d;
}
void Mailbox::Free() {
    if (host_) (void)hipHostFree(host_);
    host_ = dev_ = nullptr;
}
void Mailbox::Request(const void* src, size_t bytes, hipStream_t s) {
    KPublish<<<1, 256, 0, s>>>((const uint64_t*)src, (uint32_t)(bytes / 8), dev_ + kHeader, dev_, ++seq_);
    CGD_HIP(hipGetLastError());
}
bool Mailbox::Arrived() const {
    if (*(volatile uint64_t*)host_ != seq_) return false;
    std::atomic_thread_fence(std::memory_order_acquire);
    return true;
}
void Mailbox::Wait(hipStream_t s) const {
    // Short waits by watching; a longer one leaves the processor to others.
    const auto t0 = std::chrono::steady_clock::now();
    for (uint32_t i = 0; !Arrived(); i++) {
        if ((i & 63u) == 63u && std::chrono::steady_clock::now() - t0 > std::chrono::microseconds(200)) {
            CGD_HIP(hipStreamSynchronize(s));
            if (!Arrived()) throw HipError(hipErrorUnknown, "counter read-back", __FILE__, __LINE__);
            return;
        }
        __builtin_ia32_pause();
    }
}

size_t RadixHistWords(uint64_t n) {
    uint64_t nb = (n + kRsTile - 1) / kRsTile;
    uint64_t hn = (nb ? nb : 1) * 256;
    // histogram, one pad word, then the scan scratch of the histogram
    return (size_t)(hn + 1 + ScanScratchBytes(hn) / sizeof(uint32_t) + 2);
}

void RadixSortU64(uint64_t* keys, uint64_t* alt, uint64_t n, uint32_t bits, uint32_t* hist, hipStream_t s) {
    if (n < 2) return;
    if (n <= (uint64_t)kRsTile) {
        KRsSortTile<<<1, kBsThreads, 0, s>>>(keys, (uint32_t)n, bits);
        CGD_HIP(hipGetLastError());
        return;
    }
    const uint32_t nb = (uint32_t)((n + kRsTile - 1) / kRsTile);
    const uint64_t hn = (uint64_t)nb * 256;
    // The scan scratch lives right after the histogram.
    uint32_t* scan_scratch = hist + hn + 1;
    uint64_t* src = keys;
    uint64_t* dst = alt;
    for (uint32_t shift = 0; shift < bits; shift += 8) {
        KRsHist<<<nb, kBsThreads, 0, s>>>(src, n, shift, hist, nb);
        ScanU32(hist, hist, hn, nullptr, scan_scratch, s);
        KRsScatter<<<nb, kBsThreads, 0, s>>>(src, dst, n, shift, hist, nb);
        std::swap(src, dst);
    }
    if (src != keys) CGD_HIP(hipMemcpyAsync(keys, src, n * sizeof(uint64_t), hipMemcpyDeviceToDevice, s));
    CGD_HIP(hipGetLastError());
}

}  // namespace cgd
