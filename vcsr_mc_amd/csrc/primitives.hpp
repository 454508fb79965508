// primitives.hpp -- device-wide scan, stable LSD radix sort and small utilities, written for
// gfx950 wave64: wave scans use DPP row shifts plus v_readlane carries; the radix scatter ranks
// keys with one wave ballot per digit bit (a wave-level multisplit), so every pass is stable and
// deterministic.
#pragma once
#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <utility>

#include "device_memory.hpp"
#include "hip_common.hpp"

namespace vcsrmc {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr long long kScanTile = (long long)kScanThreads * kScanItems;

// Block-level inclusive scan of one value per thread (256 threads = 4 waves).
template <typename T, typename Op>
__device__ __forceinline__ T block_scan_256(T x, Op op, T identity, T* wsum /* LDS[4] */,
                                            T& block_total) {
    const int t = threadIdx.x, w = t >> 6;
    T incl = wave_scan(x, op, identity);
    if ((t & 63) == 63) wsum[w] = incl;
    __syncthreads();
    T wp = identity;
    for (int i = 0; i < w; ++i) wp = op(wp, wsum[i]);
    block_total = op(op(wsum[0], wsum[1]), op(wsum[2], wsum[3]));
    __syncthreads();
    return op(wp, incl);
}

// A thread's kScanItems consecutive values from index i (past n: identity), in 16-byte loads
// where all of them exist.
template <typename TIn, typename TOut>
__device__ __forceinline__ void scan_load(const TIn* __restrict__ in, long long i, long long n,
                                          TOut identity, TOut (&x)[kScanItems]) {
    constexpr int V = 16 / sizeof(TIn);
    typedef TIn vec __attribute__((ext_vector_type(V)));
    typedef vec vec_any __attribute__((aligned(sizeof(TIn))));
    if (i + kScanItems <= n) {
#pragma unroll
        for (int j = 0; j < kScanItems; j += V) {
            const vec v = *reinterpret_cast<const vec_any*>(in + i + j);
#pragma unroll
            for (int q = 0; q < V; ++q) x[j + q] = (TOut)v[q];
        }
    } else {
#pragma unroll
        for (int j = 0; j < kScanItems; ++j) x[j] = i + j < n ? (TOut)in[i + j] : identity;
    }
}

template <typename TIn, typename TOut, typename Op>
__global__ __launch_bounds__(kScanThreads) void k_reduce_tile(const TIn* __restrict__ in,
                                                              TOut* __restrict__ partial,
                                                              long long n, Op op, TOut identity) {
    __shared__ TOut wsum[4];
    TOut x[kScanItems];
    scan_load<TIn, TOut>(in, (long long)blockIdx.x * kScanTile + threadIdx.x * kScanItems, n,
                         identity, x);
    TOut acc = identity;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) acc = op(acc, x[j]);
    TOut total;
    block_scan_256(acc, op, identity, wsum, total);
    if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// EXCL: out[i] = in[0] + ... + in[i-1] (OpAdd only) and, when write_total, out[n] = total.
// Otherwise out[i] = op(in[0..i]).  A block's carry is prefix[block - 1], or (`sums`) the sum it
// takes over prefix[0 .. block - 1], the earlier tiles' totals: cheaper than the launch that would
// scan them while there are few (kScanSums).
template <typename TIn, typename TOut, typename Op, bool EXCL>
__global__ __launch_bounds__(kScanThreads) void k_scan_tile(const TIn* __restrict__ in,
                                                            TOut* __restrict__ out, long long n,
                                                            const TOut* __restrict__ prefix,
                                                            bool sums, Op op, TOut identity,
                                                            int write_total) {
    __shared__ TOut wsum[4];
    const long long i = (long long)blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    TOut x[kScanItems];
    scan_load<TIn, TOut>(in, i, n, identity, x);
    TOut carry = identity;
    if (prefix && blockIdx.x > 0) {
        if (sums) {
            TOut s = identity;
            for (unsigned b = threadIdx.x; b < blockIdx.x; b += kScanThreads) s = op(s, prefix[b]);
            block_scan_256(s, op, identity, wsum, carry);
        } else {
            carry = prefix[blockIdx.x - 1];
        }
    }
    TOut mine = identity;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) mine = op(mine, x[j]);
    TOut total;
    const TOut incl = block_scan_256(mine, op, identity, wsum, total);
    // the prefix before this thread's values: the inclusive prefix of the thread before it
    TOut run = carry;
    {
        __shared__ TOut last[kScanThreads];
        last[threadIdx.x] = incl;
        __syncthreads();
        if (threadIdx.x > 0) run = op(carry, last[threadIdx.x - 1]);
    }
    TOut y[kScanItems];
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        if constexpr (EXCL) y[j] = run;
        run = op(run, x[j]);
        if constexpr (!EXCL) y[j] = run;
    }
    constexpr int V = 16 / sizeof(TOut);
    typedef TOut vec __attribute__((ext_vector_type(V)));
    typedef vec vec_any __attribute__((aligned(sizeof(TOut))));
    if (i + kScanItems <= n) {
#pragma unroll
        for (int j = 0; j < kScanItems; j += V) {
            vec v;
#pragma unroll
            for (int q = 0; q < V; ++q) v[q] = y[j + q];
            *reinterpret_cast<vec_any*>(out + i + j) = v;
        }
    } else {
#pragma unroll
        for (int j = 0; j < kScanItems; ++j)
            if (i + j < n) out[i + j] = y[j];
    }
    if (EXCL && write_total && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0)
        out[n] = op(carry, total);
}

// Up to this many tiles, every block sums the totals of the tiles before it (at most 8 loads a
// thread) and the launch between the two passes is saved.
constexpr long long kScanSums = 2048;

template <typename TIn, typename TOut, typename Op, bool EXCL>
void scan_impl(const TIn* in, TOut* out, long long n, Op op, TOut identity, int write_total,
               hipStream_t st) {
    if (n <= 0) {
        if (EXCL && write_total) VCSRMC_HIP(hipMemsetAsync(out, 0, sizeof(TOut), st));
        return;
    }
    const long long tiles = (n + kScanTile - 1) / kScanTile;
    TmpBuf<TOut> partial(tiles > 1 ? tiles : 0), prefix(tiles > kScanSums ? tiles : 0);
    if (tiles > 1) {
        hipLaunchKernelGGL((k_reduce_tile<TIn, TOut, Op>), dim3((unsigned)tiles),
                           dim3(kScanThreads), 0, st, in, partial.p, n, op, identity);
        VCSRMC_HIP(hipGetLastError());
    }
    if (tiles > kScanSums)
        scan_impl<TOut, TOut, Op, false>(partial.p, prefix.p, tiles, op, identity, 0, st);
    hipLaunchKernelGGL((k_scan_tile<TIn, TOut, Op, EXCL>), dim3((unsigned)tiles),
                       dim3(kScanThreads), 0, st, in, out, n,
                       (const TOut*)(prefix.p ? prefix.p : partial.p), prefix.p == nullptr, op,
                       identity, write_total);
    VCSRMC_HIP(hipGetLastError());
}

// out[0..n]: exclusive prefix sums of in[0..n-1], out[n] = total.
template <typename TIn, typename TOut>
void exclusive_sum(const TIn* in, TOut* out, long long n, hipStream_t st) {
    scan_impl<TIn, TOut, OpAdd, true>(in, out, n, OpAdd{}, (TOut)0, 1, st);
}

template <typename TIn, typename TOut>
void inclusive_sum(const TIn* in, TOut* out, long long n, hipStream_t st) {
    scan_impl<TIn, TOut, OpAdd, false>(in, out, n, OpAdd{}, (TOut)0, 0, st);
}

inline void inclusive_max(const int* in, int* out, long long n, hipStream_t st) {
    scan_impl<int, int, OpMax, false>(in, out, n, OpMax{}, (int)0x80000000, 0, st);
}

// Copy one value back (synchronises the stream).
template <typename T>
T read_scalar(const T* dptr, hipStream_t st) {
    T v{};
    VCSRMC_HIP(hipMemcpyAsync(&v, dptr, sizeof(T), hipMemcpyDeviceToHost, st));
    VCSRMC_HIP(hipStreamSynchronize(st));
    return v;
}

// ---- stable LSD radix sort of keys, or (key, 32-bit payload) pairs ----------------------
// One pass: digit counts of every tile of 4096 keys, their scan, and the scatter.  Memory traffic
// bounds a pass (27 M 64-bit keys with payload: 216 MB read to count, 650 MB moved), as long as
// the scatter writes runs: each tile is put in digit order in LDS first, and consecutive threads
// then write consecutive keys of a digit.  Written straight from the registers in index order, a
// wave's 64 keys went to up to 64 places.  A pass over 27 M
// 64-bit keys with payload 697 -> 235 us at most (random columns), 64-bit keys alone 123.
constexpr int kSortThreads = 512;
constexpr int kSortWaves = kSortThreads / 64;
constexpr int kSortRounds = 8;
constexpr int kSortTile = kSortThreads * kSortRounds;

template <typename K>
__global__ __launch_bounds__(kSortThreads) void k_radix_hist(const K* __restrict__ keys, long long n,
                                                             int shift, int digits,
                                                             int* __restrict__ hist, int ntiles) {
    __shared__ int h[256];
    if (threadIdx.x < 256) h[threadIdx.x] = 0;
    __syncthreads();
    const long long base = (long long)blockIdx.x * kSortTile;
    K key[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const long long i = base + r * kSortThreads + threadIdx.x;
        key[r] = i < n ? keys[i] : (K)0;
    }
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const long long i = base + r * kSortThreads + threadIdx.x;
        if (i < n) atomicAdd(&h[(int)(key[r] >> shift) & (digits - 1)], 1);
    }
    __syncthreads();
    if (threadIdx.x < digits) hist[(long long)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

// offsets: exclusive scan of the digit-major histogram.  Keys of one tile are ranked in index
// order: wave w ranks the tile's keys 64 w R .. 64 (w + 1) R - 1 (R rounds of 64, lanes by ballot
// multisplit, rounds by the wave's running digit counts), then waves in order; tiles were ordered
// by the scan.
template <typename K, bool VAL>
__global__ __launch_bounds__(kSortThreads) void k_radix_scatter(
    const K* __restrict__ kin, const uint32_t* __restrict__ vin, K* __restrict__ kout,
    uint32_t* __restrict__ vout, long long n, int shift, int bits, const int* __restrict__ offsets,
    int ntiles) {
    __shared__ int wcnt[kSortWaves][256];  // per wave: digit counts, then first place in the tile
    __shared__ int gofs[256];              // where the tile's digit goes, less its place here
    __shared__ int wsum[4];
    __shared__ K skey[kSortTile];
    __shared__ uint32_t sval[VAL ? kSortTile : 1];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const int mask = (1 << bits) - 1;
    for (int i = t; i < kSortWaves * 256; i += kSortThreads) (&wcnt[0][0])[i] = 0;
    const long long base = (long long)blockIdx.x * kSortTile;
    const int count = (int)min((long long)kSortTile, n - base);
    const int first = w * 64 * kSortRounds + lane;
    K key[kSortRounds];
    uint32_t val[VAL ? kSortRounds : 1];
    int rank[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const int i = first + r * 64;
        key[r] = i < count ? kin[base + i] : (K)0;
        if constexpr (VAL) val[r] = i < count ? vin[base + i] : 0u;
    }
    __syncthreads();
    const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const bool valid = first + r * 64 < count;
        const int d = (int)(key[r] >> shift) & mask;
        uint64_t peers = __ballot(valid);
        for (int b = 0; b < bits; ++b) {
            const bool bit = (d >> b) & 1;
            const uint64_t m = __ballot(bit);
            peers &= bit ? m : ~m;
        }
        const int before = wcnt[w][d], in_round = __popcll(peers & below);
        rank[r] = before + in_round;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (valid && in_round == 0) wcnt[w][d] = before + __popcll(peers);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __syncthreads();
    // thread t < 256: the tile's count of digit t; a scan over the four waves that hold them
    int total = 0, incl = 0;
    if (t < 256) {
#pragma unroll
        for (int i = 0; i < kSortWaves; ++i) total += wcnt[i][t];
        incl = wave_scan(total, OpAdd{}, 0);
        if (lane == 63) wsum[w] = incl;
    }
    __syncthreads();
    if (t < 256) {
        int start = incl - total;
        for (int i = 0; i < w; ++i) start += wsum[i];
        if (t <= mask) gofs[t] = offsets[(long long)t * ntiles + blockIdx.x] - start;
#pragma unroll
        for (int i = 0; i < kSortWaves; ++i) {
            const int c = wcnt[i][t];
            wcnt[i][t] = start;
            start += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r)
        if (first + r * 64 < count) {
            const int at = wcnt[w][(int)(key[r] >> shift) & mask] + rank[r];
            skey[at] = key[r];
            if constexpr (VAL) sval[at] = val[r];
        }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const int i = r * kSortThreads + t;
        if (i < count) {
            const K k = skey[i];
            const int dst = gofs[(int)(k >> shift) & mask] + i;
            kout[dst] = k;
            if constexpr (VAL) vout[dst] = sval[i];
        }
    }
}

// Passes of equal width, at most 8 bits each: the first reads (src, vsrc), the others what the
// pass before wrote, in (a, va) and (b, vb) by turns.  Returns the sorted keys and payload.
template <typename K, bool VAL>
std::pair<K*, uint32_t*> radix_sort_impl(const K* src, const uint32_t* vsrc, K* a, uint32_t* va,
                                         K* b, uint32_t* vb, long long n, int bits,
                                         hipStream_t st) {
    const int passes = (bits + 7) / 8, width = (bits + passes - 1) / passes;
    const int ntiles = (int)((n + kSortTile - 1) / kSortTile);
    TmpBuf<int> hist((size_t)ntiles << width), offs(((size_t)ntiles << width) + 1);
    for (int shift = 0; shift < bits; shift += width) {
        hipLaunchKernelGGL((k_radix_hist<K>), dim3(ntiles), dim3(kSortThreads), 0, st, src, n,
                           shift, 1 << width, hist.p, ntiles);
        VCSRMC_HIP(hipGetLastError());
        exclusive_sum<int, int>(hist.p, offs.p, (long long)ntiles << width, st);
        hipLaunchKernelGGL((k_radix_scatter<K, VAL>), dim3(ntiles), dim3(kSortThreads), 0, st, src,
                           vsrc, a, va, n, shift, width, offs.p, ntiles);
        VCSRMC_HIP(hipGetLastError());
        src = a;
        vsrc = va;
        std::swap(a, b);
        std::swap(va, vb);
    }
    return {b, vb};
}

// The n pairs of (src, vsrc), which stay as they are, sorted by the low `bits` (>= 1) bits of the
// key into one of the two given pairs of arrays, the other being scratch.  n must be below 2^31.
template <typename K>
std::pair<K*, uint32_t*> radix_sort_pairs_from(const K* src, const uint32_t* vsrc, K* a,
                                               uint32_t* va, K* b, uint32_t* vb, long long n,
                                               int bits, hipStream_t st) {
    return radix_sort_impl<K, true>(src, vsrc, a, va, b, vb, n, bits, st);
}

// Sorts n pairs by the low `bits` bits of the key.  The sorted pairs end up in (k, v); the
// alternate buffers are scratch of the same size.  n must be below 2^31.
template <typename K>
void radix_sort_pairs(K*& k, uint32_t*& v, K*& k_alt, uint32_t*& v_alt, long long n, int bits,
                      hipStream_t st) {
    if (n <= 1 || bits <= 0) return;
    const auto out = radix_sort_impl<K, true>(k, v, k_alt, v_alt, k, v, n, bits, st);
    if (out.first != k) {
        std::swap(k, k_alt);
        std::swap(v, v_alt);
    }
}

// The same for keys alone.
template <typename K>
void radix_sort_keys(K*& k, K*& k_alt, long long n, int bits, hipStream_t st) {
    if (n <= 1 || bits <= 0) return;
    const auto out = radix_sort_impl<K, false>(k, nullptr, k_alt, nullptr, k, nullptr, n, bits, st);
    if (out.first != k) std::swap(k, k_alt);
}

// ---- small kernels -----------------------------------------------------------------------
template <typename T>
__global__ void k_fill(T* __restrict__ p, long long n, T value) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

template <typename T>
void fill(T* p, long long n, T value, hipStream_t st) {
    if (n <= 0) return;
    hipLaunchKernelGGL((k_fill<T>), dim3(grid_for(n, 256)), dim3(256), 0, st, p, n, value);
    VCSRMC_HIP(hipGetLastError());
}

// ptr[v] = the first index of the ascending `keys` (each below count) that is >= v, for v in
// [0, count]: every change of the key writes the values it passes, the whole wave where they are
// many.
__device__ __forceinline__ void key_ptr_write(int from, int to, int i, int* __restrict__ ptr) {
    uint64_t wide = __ballot(to - from >= 64);
    if (to - from < 64)
        for (int v = from; v <= to; ++v) ptr[v] = i;
    while (wide) {
        const int l = (int)__builtin_ctzll(wide);
        wide &= wide - 1;
        const int f = __shfl(from, l), t = __shfl(to, l), x = __shfl(i, l);
        for (int v = f + (int)(threadIdx.x & 63); v <= t; v += 64) ptr[v] = x;
    }
}

template <typename K>
__global__ __launch_bounds__(256) void k_key_ptr(const K* __restrict__ keys, long long n,
                                                 int count, int* __restrict__ ptr) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    int from = 1, to = 0;  // nothing to write
    if (i <= n) {
        from = i == 0 ? 0 : (int)keys[i - 1] + 1;
        to = i == n ? count : (int)keys[i];
    }
    key_ptr_write(from, to, (int)i, ptr);
}

template <typename K>
void key_ptr(const K* keys, long long n, int count, int* ptr, hipStream_t st) {
    hipLaunchKernelGGL((k_key_ptr<K>), dim3(grid_for(n + 1, 256)), dim3(256), 0, st, keys, n, count,
                       ptr);
    VCSRMC_HIP(hipGetLastError());
}

}  // namespace vcsrmc
