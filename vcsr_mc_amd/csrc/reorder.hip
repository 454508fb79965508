// reorder.hip -- reverse Cuthill-McKee column order and the column relabelling that goes with
// it, on the GPU (include/reorder.hpp:17-108 of MuuSeoTia/VCSR_MC).
//
// The reference walks the symmetrised pattern breadth-first with one host queue.  Here the
// same order is produced level by level, every connected component at once:
//   1. adjacency: the 2 nnz (vertex, neighbour) pairs of the symmetrised pattern, radix-sorted
//      and deduplicated; the degree counts distinct neighbours, a self-loop included
//      (reorder.hpp:21-42).
//   2. rank: vertices in ascending (degree, id) -- the reference's stable_sort of the roots
//      (reorder.hpp:47-50).
//   3. components: rounds of hooking (the parent of larger rank under the parent of smaller
//      rank, across every edge between two trees) and pointer jumping, until a round changes
//      nothing; each component ends up represented by its lowest-rank vertex, the root from
//      which the reference's loop (reorder.hpp:54-57) starts that component.
//   4. levels: level 0 holds every component's root in rank order.  A vertex of level L+1
//      belongs to the earliest level-L vertex adjacent to it (the one that pops it from the
//      reference's queue, reorder.hpp:63-66).  A level is ordered by that parent's index, then
//      inside one parent's children as the reference orders them: ascending id, then
//      std::sort by degree (reorder.hpp:67-69), whose steps (libstdc++ introsort) are carried
//      out exactly, since equal degrees make the result depend on them.  Levels of up to 8192
//      frontier edges run inside one work-group, many at a time (k_bfs_levels); larger ones take
//      four kernels each over the frontier's edges (k_level_claim, _count, _place, _sort), with
//      their sizes kept on the device, so that several levels are enqueued at a time.
//   5. order: vertices sorted by (component rank, place in the walk) give the
//      Cuthill-McKee order; position = N - 1 - that index (reorder.hpp:72-76).
#include <algorithm>
#include <atomic>
#include <climits>
#include <cstdint>
#include <string>
#include <type_traits>

#include "../../include/vcsrmc.h"
#include "internal.hpp"

namespace vcsrmc {
namespace {

using u64 = unsigned long long;

inline unsigned nblk(long long n) { return grid_for(n, 256); }

#define RLAUNCH(kernel, n, ...)                                                               \
    do {                                                                                      \
        if ((n) > 0) {                                                                        \
            hipLaunchKernelGGL(kernel, dim3(nblk(n)), dim3(256), 0, st, __VA_ARGS__);         \
            VCSRMC_HIP(hipGetLastError());                                                    \
        }                                                                                     \
    } while (0)

enum : int { kBadRowPtr = 1, kBadCol = 2, kBadPerm = 4, kDupCol = 8 };

__global__ void k_check_rp(const int* __restrict__ rp, int M, int nnz, int* __restrict__ err) {
    const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r > M) return;
    const int a = rp[r];
    bool bad = a < 0 || a > nnz;
    if (r == 0) bad |= a != 0;
    if (r == M) bad |= a != nnz;
    if (r < M) bad |= rp[r + 1] < a;
    if (bad) atomicOr(err, kBadRowPtr);
}

__global__ void k_check_cols(const int* __restrict__ col, long long nnz, int N,
                             int* __restrict__ err) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnz) return;
    const int c = col[i];
    if (c < 0 || c >= N) atomicOr(err, kBadCol);
}

void raise_if(const int* d_err, hipStream_t st) {
    const int e = read_scalar(d_err, st);
    if (e & kBadRowPtr) throw Error(VCSRMC_ERR_CSR, "row_ptr is not a monotone 0..nnz sequence");
    if (e & kBadCol) throw Error(VCSRMC_ERR_CSR, "column index out of range [0, N)");
    if (e & kBadPerm) throw Error(VCSRMC_ERR_ARG, "position is not a permutation of 0..N-1");
    if (e & kDupCol)
        throw Error(VCSRMC_ERR_UNSORTED, "a row holds the same column twice");
}

void check_csr(const int* rp, const int* col, int M, int N, int nnz, int* d_err, hipStream_t st) {
    VCSRMC_HIP(hipMemsetAsync(d_err, 0, sizeof(int), st));
    RLAUNCH(k_check_rp, (long long)M + 1, rp, M, nnz, d_err);
    RLAUNCH(k_check_cols, (long long)nnz, col, (long long)nnz, N, d_err);
    raise_if(d_err, st);
}

// ---- 1. adjacency ------------------------------------------------------------------------
// Nonzero (r, c) contributes r -> c and c -> r when r < N; a row r >= N has no vertex of its
// own and makes c its own neighbour (twice, merged by the deduplication).
template <typename K>
__global__ void k_adj_pairs(const int* __restrict__ row_of, const int* __restrict__ col,
                            long long nnz, int N, int nb, K* __restrict__ key) {
    typedef K pair __attribute__((ext_vector_type(2)));
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nnz) return;
    const int r = row_of[p], c = col[p];
    const bool own = r < N;
    const K first = own ? ((K)r << nb | (K)c) : ((K)c << nb | (K)c);
    *reinterpret_cast<pair*>(key + 2 * p) = pair{first, (K)c << nb | (K)(own ? r : c)};
}

template <typename K>
__global__ void k_unique_flags(const K* __restrict__ key, long long n, int* __restrict__ flag) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) flag[i] = (i == 0 || key[i] != key[i - 1]) ? 1 : 0;
}

template <typename K>
__global__ void k_unique_write(const K* __restrict__ key, const int* __restrict__ pos, long long n,
                               int nb, int* __restrict__ adj_u, int* __restrict__ adj) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || pos[i + 1] == pos[i]) return;
    const K k = key[i];
    const int p = pos[i];
    adj_u[p] = (int)(k >> nb);
    adj[p] = (int)(k & (((K)1 << nb) - 1));
}

// ---- 2. rank -----------------------------------------------------------------------------
// Degrees; the stable sort keeps vertices of one degree by id.
__global__ void k_rank_keys(const int* __restrict__ head, int N, uint32_t* __restrict__ key,
                            uint32_t* __restrict__ val) {
    const long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= N) return;
    key[v] = (uint32_t)(head[v + 1] - head[v]);
    val[v] = (uint32_t)v;
}

__global__ void k_scatter_rank(const uint32_t* __restrict__ order, int N, int* __restrict__ rank) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) rank[order[i]] = (int)i;
}

// ---- 3. components -----------------------------------------------------------------------
// Rounds of hooking and pointer jumping over plain loads and stores.  A round hooks, for every
// edge whose ends have different parents, the parent of larger rank under the other one if it
// is still a root, then moves every vertex to its grandparent.  parent[] only ever points to a
// vertex of smaller rank, so the trees stay acyclic whatever order the stores land in.  A round
// that changes nothing leaves every tree a star (each vertex's parent is a root) and no edge
// between two trees, so parent[v] is then the root of v's component, its lowest-rank vertex:
// the vertex the reference's loop over roots in rank order starts the component from.
__global__ void k_cc_init(int* __restrict__ parent, int N) {
    const long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v < N) parent[v] = (int)v;
}

__global__ void k_cc_hook(const int* __restrict__ adj_u, const int* __restrict__ adj, long long E,
                          const int* __restrict__ rank, int* parent, int* __restrict__ changed) {
    const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    const int u = adj_u[e], w = adj[e];
    if (u >= w) return;  // each undirected edge once; self-loops join nothing
    int a = parent[u], b = parent[w];
    if (a == b) return;
    if (rank[a] > rank[b]) { const int t = a; a = b; b = t; }
    if (parent[b] == b) {
        parent[b] = a;
        *changed = 1;
    }
}

__global__ void k_cc_jump(int* parent, int N, int* __restrict__ changed) {
    const long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= N) return;
    const int p = parent[v], gp = parent[p];
    if (gp != p) {
        parent[v] = gp;
        *changed = 1;
    }
}

// ---- 4. levels ---------------------------------------------------------------------------
__global__ void k_root_flags(const uint32_t* __restrict__ order, const int* __restrict__ comp,
                             int N, int* __restrict__ flag) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) flag[i] = comp[order[i]] == (int)order[i] ? 1 : 0;
}

__global__ void k_root_list(const uint32_t* __restrict__ order, const int* __restrict__ flag,
                            const int* __restrict__ pos, int N, int* __restrict__ walk,
                            int* __restrict__ seq) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N || !flag[i]) return;
    const int v = (int)order[i];
    const int p = pos[i];
    walk[p] = v;
    seq[v] = p;
}

// std::sort(first, last, [](a, b) { return degree[a] < degree[b]; }) with the steps of GCC 11's
// libstdc++ (introsort: median-of-three Hoare partitions while a range holds more than 16
// elements, heapsort once 2 floor(lg n) partition levels are used up, then one insertion pass).
// The scans carry bounds checks the library omits; they never fire, as the median-of-three
// pivot and the insertion pass's leftmost minimum stop every scan inside its range.
__device__ __forceinline__ uint32_t skey(u64 x) { return (uint32_t)(x >> 32); }

__device__ void ls_insert(u64* a, long long lo, long long pos) {
    const u64 v = a[pos];
    while (pos > lo && skey(v) < skey(a[pos - 1])) {
        a[pos] = a[pos - 1];
        --pos;
    }
    a[pos] = v;
}

__device__ void ls_sift(u64* a, long long base, long long hole, long long len, u64 v) {
    const long long top = hole;
    long long child = hole;
    while (child < (len - 1) / 2) {
        child = 2 * child + 2;
        if (skey(a[base + child]) < skey(a[base + child - 1])) --child;
        a[base + hole] = a[base + child];
        hole = child;
    }
    if ((len & 1) == 0 && child == (len - 2) / 2) {
        child = 2 * child + 2;
        a[base + hole] = a[base + child - 1];
        hole = child - 1;
    }
    long long parent = (hole - 1) / 2;
    while (hole > top && skey(a[base + parent]) < skey(v)) {
        a[base + hole] = a[base + parent];
        hole = parent;
        parent = (hole - 1) / 2;
    }
    a[base + hole] = v;
}

__device__ void ls_heapsort(u64* a, long long lo, long long hi) {
    const long long len = hi - lo;
    if (len >= 2)
        for (long long parent = (len - 2) / 2;; --parent) {
            ls_sift(a, lo, parent, len, a[lo + parent]);
            if (parent == 0) break;
        }
    for (long long end = hi - 1; end - lo > 0; --end) {
        const u64 v = a[end];
        a[end] = a[lo];
        ls_sift(a, lo, 0, end - lo, v);
    }
}

__device__ __forceinline__ void ls_swap(u64* a, long long i, long long j) {
    const u64 t = a[i];
    a[i] = a[j];
    a[j] = t;
}

__device__ void ls_median_to_first(u64* a, long long dst, long long x, long long y, long long z) {
    const uint32_t kx = skey(a[x]), ky = skey(a[y]), kz = skey(a[z]);
    if (kx < ky) {
        if (ky < kz) ls_swap(a, dst, y);
        else if (kx < kz) ls_swap(a, dst, z);
        else ls_swap(a, dst, x);
    } else if (kx < kz) {
        ls_swap(a, dst, x);
    } else if (ky < kz) {
        ls_swap(a, dst, z);
    } else {
        ls_swap(a, dst, y);
    }
}

// Every pass moves lo up and hi down by at least one, so at most (hi - lo) / 2 + 1 passes run;
// the loop states that bound.
__device__ long long ls_partition(u64* a, long long lo, long long hi, long long piv) {
    const uint32_t kp = skey(a[piv]);
    const long long end = hi;
    for (long long pass = (hi - lo) / 2 + 1; pass >= 0; --pass) {
        while (lo < end && skey(a[lo]) < kp) ++lo;
        --hi;
        while (hi > piv && kp < skey(a[hi])) --hi;
        if (!(lo < hi)) return lo;
        ls_swap(a, lo, hi);
        ++lo;
    }
    return lo;
}

struct SortRange {
    int lo, hi, depth;
};

// std::sort's introsort loop on a[lo, hi) from partition depth `depth`, then its insertion
// pass over the same range.  Ranges that the loop leaves untouched are independent, so any
// subrange the partitions produce can be finished on its own: the insertion pass never moves
// an element across a partition boundary (left part <= pivot <= right part, and it only moves
// past strictly greater keys).
__device__ void ls_sort_range(u64* a, int lo0, int hi0, int depth0) {
    if (hi0 - lo0 <= 1) return;
    SortRange stack[64];
    int sp = 0;
    stack[sp++] = {lo0, hi0, depth0};
    while (sp > 0) {
        const SortRange r = stack[--sp];
        long long lo = r.lo, hi = r.hi;
        int depth = r.depth;
        while (hi - lo > 16) {
            if (depth == 0) {
                ls_heapsort(a, lo, hi);
                break;
            }
            --depth;
            ls_median_to_first(a, lo, lo + 1, lo + (hi - lo) / 2, hi - 1);
            const long long cut = ls_partition(a, lo + 1, hi, lo);
            if (sp < 64) stack[sp++] = {(int)cut, (int)hi, depth};
            hi = cut;
        }
    }
    for (int i = lo0 + 1; i < hi0; ++i) ls_insert(a, lo0, i);
}

__device__ __forceinline__ int lg_floor(int n) {
    int lg = 0;
    while ((2ll << lg) <= n) ++lg;
    return lg;
}

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The walk.  walk[i] = the vertex of place i, seq[v] = v's place or -1; a level's frontier is the
// last f vertices placed.  state = {frontier size, vertices placed, level, finished}.  A vertex
// reached from several frontier vertices belongs to the one of the lowest place: claim[u] = the
// smallest place of a frontier vertex adjacent to u, taken only while u has no place, so
// claim[u] == place tells a parent its children, in every later kernel of the level.
//
// ---- 4a. small levels in one work-group ---------------------------------------------------
// While a level has at most kBfsCap frontier vertices and frontier edges, one work-group runs
// level after level with no host round trip: each frontier edge claims its neighbour, then an
// edge holds a child when its frontier vertex won the claim.  Frontier vertices are in level order
// and each adjacency list is in ascending id, so an exclusive scan over the edges places the
// children in (parent index, ascending id) order directly; each parent's children are then sorted
// by degree with std::sort's steps in LDS: groups of up to kBfsSortSmall by their parent's thread,
// larger ones (the children of hub vertices) partitioned by the whole work-group, a step at a
// time, and the pieces finished by one thread each.  Thread t owns a contiguous run of up to
// kBfsPer vertices or edges, so each phase needs one block scan.  The work-group stops at the
// first level that does not fit (state.w = 0) or when the walk ends (state.w = 1).
constexpr int kBfsThreads = 1024;
constexpr int kBfsPer = 8;
constexpr int kBfsCap = kBfsThreads * kBfsPer;
constexpr int kBfsSortSmall = 64;
constexpr int kBfsMaxBig = kBfsCap / (kBfsSortSmall + 1) + 1;
// Marks of the piece starts during the work-group sort (one byte per child position): the
// partition depth a piece continues from, or one of these.
constexpr unsigned char kMarkNone = 255, kMarkGroupEnd = 254, kMarkHeap = 253;

template <int NW>
__device__ __forceinline__ int block_scan_int(int x, int* wsum /* LDS[NW] */, int& total) {
    const int t = threadIdx.x, w = t >> 6;
    const int incl = wave_scan(x, OpAdd{}, 0);
    if ((t & 63) == 63) wsum[w] = incl;
    __syncthreads();
    int before = 0, all = 0;
    for (int i = 0; i < NW; ++i) {
        const int s = wsum[i];
        if (i < w) before += s;
        all += s;
    }
    total = all;
    __syncthreads();
    return before + incl;
}

template <int NW>
__device__ __forceinline__ void team_sync() {
    if constexpr (NW == 1) wave_lds_fence();
    else __syncthreads();
}

// One step of the introsort loop on a[lo, hi) (depth > 0), in LDS or memory, by NW waves (one: a
// wave on its own; more: the whole work-group), with the same result as the library's sequential
// step.  After the median of three is moved to a[lo], the Hoare scans over a[lo+1, hi) stop, from
// the left, at elements whose key is not below the pivot's (l_1 < l_2 < ...) and, from the right,
// at elements whose key is not above it (r_1 > r_2 > ...); the k-th swap exchanges a[l_k] and
// a[r_k] while l_k < r_k, so K = the number of left stops x with at least rank(x) right stops
// after x; the cut is l_1 when K = 0, else min(l_{K+1}, r_K).  Both parts continue with depth - 1;
// a range at depth 0 is heapsorted.  Each wave counts and ranks a run of its own by ballots.
// lpos and rpos hold the pair positions (K <= (hi - lo) / 2, as the pairs are disjoint); part (NW
// entries) and lnext are LDS of the team.  Returns the cut (the same value in every thread).
template <int NW>
__device__ int partition_step(u64* a, int lo, int hi, int* lpos, int* rpos, int2* part,
                              int* lnext) {
    const int lane = threadIdx.x & 63, w = NW == 1 ? 0 : (int)(threadIdx.x >> 6);
    const int t = NW == 1 ? lane : (int)threadIdx.x;
    if (t == 0) {
        ls_median_to_first(a, lo, lo + 1, lo + (hi - lo) / 2, hi - 1);
        *lnext = INT_MAX;
    }
    team_sync<NW>();
    const uint32_t kp = skey(a[lo]);
    const int first = lo + 1, n = hi - first;
    const int per = ((n + NW - 1) / NW + 63) / 64 * 64;
    const int b0 = min(first + w * per, hi), b1 = min(b0 + per, hi);
    const u64 below = lane ? (~0ull >> (64 - lane)) : 0ull;
    // masks of the left and right stops among the 64 elements at p
    const auto stops = [&](int p, u64& ge, u64& le) {
        const bool in = p + lane < b1;
        const uint32_t k = in ? skey(a[p + lane]) : 0u;
        ge = __ballot(in && !(k < kp));
        le = __ballot(in && !(kp < k));
    };
    u64 ge, le;
    int cge = 0, cle = 0;
    for (int p = b0; p < b1; p += 64) {
        stops(p, ge, le);
        cge += __popcll(ge);
        cle += __popcll(le);
    }
    int ge_before = 0, le_before = 0, LE = cle;
    if constexpr (NW > 1) {
        if (lane == 0) part[w] = make_int2(cge, cle);
        __syncthreads();
        LE = 0;
        for (int i = 0; i < NW; ++i) {
            const int2 x = part[i];
            ge_before += i < w ? x.x : 0;
            le_before += i < w ? x.y : 0;
            LE += x.y;
        }
        __syncthreads();
    }
    int K = 0;
    {
        int g = ge_before, l = le_before;
        for (int p = b0; p < b1; p += 64) {
            stops(p, ge, le);
            const int rank = g + __popcll(ge & below) + 1;
            const int le_incl = l + __popcll(le & below) + (int)((le >> lane) & 1);
            K += __popcll(__ballot(((ge >> lane) & 1) && LE - le_incl >= rank));
            g += __popcll(ge);
            l += __popcll(le);
        }
    }
    if constexpr (NW > 1) {
        if (lane == 0) part[w].x = K;
        __syncthreads();
        K = 0;
        for (int i = 0; i < NW; ++i) K += part[i].x;
    }
    {
        int g = ge_before, l = le_before;
        for (int p = b0; p < b1; p += 64) {
            stops(p, ge, le);
            if ((ge >> lane) & 1) {
                const int rank = g + __popcll(ge & below) + 1;
                if (rank <= K) lpos[rank - 1] = p + lane;
                else if (rank == K + 1) *lnext = p + lane;
            }
            if ((le >> lane) & 1) {
                const int rr = LE - (l + __popcll(le & below));
                if (rr <= K) rpos[rr - 1] = p + lane;
            }
            g += __popcll(ge);
            l += __popcll(le);
        }
    }
    team_sync<NW>();
    for (int r = t; r < K; r += 64 * NW) {
        const int x = lpos[r], y = rpos[r];
        const u64 ax = a[x], ay = a[y];
        a[x] = ay;
        a[y] = ax;
    }
    const int cut = K == 0 ? *lnext : min(*lnext, rpos[K - 1]);
    team_sync<NW>();
    return cut;
}

// The partition steps of std::sort on a[lo, hi) from partition depth `depth`: leaf(lo, hi, depth)
// for every piece of at most `stop` elements, or of any size with the depth used up.
// Every thread runs the same stack of ranges (lo, hi, depth) in its own registers: its control flow
// depends only on values all threads share (the ranges and the cuts), and no branch taken by one
// thread alone decides what the others do next (with the stack in LDS and thread 0 alone updating
// it, the compiler moved that update out of the loop for thread 0, and the other threads never saw
// it).
template <int NW, typename Leaf>
__device__ void partition_range(u64* a, int lo, int hi, int depth, int stop, int* lpos, int* rpos,
                                int2* part, int* lnext, Leaf&& leaf) {
    int4 stk[64];  // depth <= 2 floor(lg n) <= 62 for n < 2^31
    int sp = 1;
    stk[0] = make_int4(lo, hi, depth, 0);
    while (sp > 0) {
        const int4 r = stk[sp - 1];
        if (r.y - r.x <= stop || r.z == 0) {
            leaf(r.x, r.y, r.z);
            --sp;
        } else {
            const int cut = partition_step<NW>(a, r.x, r.y, lpos, rpos, part, lnext);
            stk[sp - 1] = make_int4(cut, r.y, r.z - 1, 0);
            stk[sp] = make_int4(r.x, cut, r.z - 1, 0);
            ++sp;
        }
    }
}

// Sorting a group in LDS takes three widths: the work-group partitions ranges down to kWavePiece
// elements, each wave partitions pieces that start in its part of the array down to kBfsSortSmall,
// and one thread finishes each of those.  mark[i] (one byte an element) says what starts at i: the
// partition depth a piece continues from, or one of the marks above.
constexpr int kWavePiece = 512;

template <int NW>
__device__ void mark_group(u64* a, int lo, int hi, int depth, unsigned char* mark, int* lpos,
                           int* rpos, int2* part, int* lnext) {
    partition_range<NW>(a, lo, hi, depth, kWavePiece, lpos, rpos, part, lnext,
                        [&](int x, int y, int d) {
                            mark[x] = y - x > kWavePiece ? kMarkHeap : (unsigned char)d;
                        });
}

// Pieces of a[0, n) (n <= kBfsCap) above kBfsSortSmall elements partitioned by waves; lnext: one
// LDS word a wave.  Each wave notes the pieces that start in its part before any wave marks more.
template <int NW>
__device__ void wave_pieces(u64* a, int n, unsigned char* mark, int* lpos, int* rpos, int* lnext) {
    constexpr int P = kBfsCap / NW / 64;
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, base = w * P * 64;
    u64 starts[P];
#pragma unroll
    for (int k = 0; k < P; ++k) {
        const int i = base + 64 * k + lane;
        starts[k] = __ballot(i < n && mark[i] < kMarkHeap);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < P; ++k) {
        while (starts[k]) {
            const int lo = base + 64 * k + (int)__builtin_ctzll(starts[k]);
            starts[k] &= starts[k] - 1;
            int hi = lo + 1;  // the next mark, or n
            for (;;) {
                const u64 m = __ballot(hi + lane >= n || mark[hi + lane] != kMarkNone);
                if (m) {
                    hi += (int)__builtin_ctzll(m);
                    break;
                }
                hi += 64;
            }
            if (hi - lo <= kBfsSortSmall) continue;
            partition_range<1>(a, lo, hi, (int)mark[lo], kBfsSortSmall, lpos + lo / 2,
                               rpos + lo / 2, nullptr, lnext + w, [&](int x, int y, int d) {
                                   mark[x] = y - x > kBfsSortSmall ? kMarkHeap : (unsigned char)d;
                               });
        }
    }
    __syncthreads();
}

// Finishes the marked pieces of a[lo, hi): std::sort's insertion pass, or its heapsort.
__device__ void finish_pieces(u64* a, int lo, int hi, const unsigned char* mark) {
    for (int i = lo + (int)threadIdx.x; i < hi; i += kBfsThreads) {
        const int m = mark[i];
        if (m > kMarkHeap) continue;
        int e = i + 1;
        while (e < hi && mark[e] == kMarkNone) ++e;  // the group's end is marked
        if (m == kMarkHeap) ls_heapsort(a, i, e);    // depth exhausted
        else if (e - i > 1) ls_sort_range(a, i, e, m);
    }
}

// A walk of N vertices has at most N levels after the roots; the loop runs to `max_level` at
// most (N + 1, or lower when a test asks) and otherwise reports state.w = kBfsOverrun.
constexpr int kBfsOverrun = 2;

__global__ __launch_bounds__(kBfsThreads) void k_bfs_levels(
    int* __restrict__ walk, const int* __restrict__ head, const int* __restrict__ adj,
    int* __restrict__ seq, int* claim, int N, long long max_level, int4* __restrict__ state) {
    constexpr int NW = kBfsThreads / 64;
    __shared__ int s_ofs[kBfsCap + 1];    // edge offset of each frontier vertex
    __shared__ int s_fx[kBfsCap + 1];     // the frontier; then children before each edge
    __shared__ u64 s_packed[kBfsCap];     // degree << 32 | id of the next level
    __shared__ int s_wsum[NW];
    __shared__ int2 s_big[kBfsMaxBig];  // child groups larger than kBfsSortSmall
    __shared__ int s_nbig, s_lnext[NW];
    __shared__ int2 s_part[NW];
    int* const s_front = s_fx;
    int* const s_ex = s_fx;
    unsigned char* const s_mark = reinterpret_cast<unsigned char*>(s_fx);  // during the sort
    const int t = threadIdx.x;
    const int4 s0 = *state;
    int f = s0.x, base = s0.y, level = s0.z;
    if (s0.w || f > kBfsCap) return;
    bool finished = false, overrun = false;
    for (int i = t; i < f; i += kBfsThreads) s_front[i] = walk[base - f + i];
    // `level` is the same in every thread: the bound ends the loop for all of them at once.
    for (;;) {
        __syncthreads();
        if (f == 0 || base >= N) {
            finished = true;
            break;
        }
        if (level > max_level) {
            overrun = true;
            break;
        }
        // edge offsets of the frontier vertices [v0, v1) of this thread
        const int pf = (f + kBfsThreads - 1) / kBfsThreads;
        const int v0 = min(t * pf, f), v1 = min(v0 + pf, f);
        int deg[kBfsPer];
        int dsum = 0;
#pragma unroll
        for (int i = 0; i < kBfsPer; ++i) {
            deg[i] = 0;
            if (v0 + i < v1) {
                const int v = s_front[v0 + i];
                deg[i] = min(head[v + 1] - head[v], kBfsCap + 1);
                dsum += deg[i];
            }
        }
        int Ef;
        int ofs = block_scan_int<NW>(dsum, s_wsum, Ef) - dsum;
        if (Ef == 0) {
            finished = true;
            break;
        }
        if (Ef > kBfsCap) break;
#pragma unroll
        for (int i = 0; i < kBfsPer; ++i)
            if (v0 + i < v1) {
                s_ofs[v0 + i] = ofs;
                ofs += deg[i];
            }
        if (t == 0) s_ofs[f] = Ef;
        __syncthreads();
        // claims of the edges [e0, e1) of this thread
        const int pe = (Ef + kBfsThreads - 1) / kBfsThreads;
        const int e0 = min(t * pe, Ef), e1 = min(e0 + pe, Ef);
        int us[kBfsPer], los[kBfsPer];
        {
            int lo = 0, hi = f;  // largest lo with s_ofs[lo] <= e0
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (s_ofs[mid] <= e0) lo = mid;
                else hi = mid;
            }
#pragma unroll
            for (int i = 0; i < kBfsPer; ++i) {
                us[i] = -1;
                los[i] = 0;
                const int e = e0 + i;
                if (e < e1) {
                    while (s_ofs[lo + 1] <= e) ++lo;
                    const int v = s_front[lo];
                    const int u = adj[head[v] + (e - s_ofs[lo])];
                    if (seq[u] < 0) {
                        los[i] = base - f + lo;
                        atomicMin(&claim[u], los[i]);
                        us[i] = u;
                    }
                }
            }
        }
        __syncthreads();
        int child = 0, nchild = 0;
#pragma unroll
        for (int i = 0; i < kBfsPer; ++i) {
            const bool c = us[i] >= 0 && __hip_atomic_load(claim + us[i], __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_AGENT) == los[i];
            child |= (int)c << i;
            nchild += c;
        }
        int n;
        int pos = block_scan_int<NW>(nchild, s_wsum, n) - nchild;
#pragma unroll
        for (int i = 0; i < kBfsPer; ++i)
            if (e0 + i < e1) {
                s_ex[e0 + i] = pos;
                if ((child >> i) & 1) {
                    const int u = us[i];
                    s_packed[pos++] = (u64)(head[u + 1] - head[u]) << 32 | (u64)(uint32_t)u;
                }
            }
        if (t == 0) {
            s_ex[Ef] = n;
            s_nbig = 0;
        }
        __syncthreads();
        for (int lo = v0; lo < v1; ++lo) {
            const int b = s_ex[s_ofs[lo]], e = s_ex[s_ofs[lo + 1]];
            if (e - b > kBfsSortSmall) s_big[atomicAdd(&s_nbig, 1)] = make_int2(b, e);
            else if (e - b > 1) ls_sort_range(s_packed, b, e, 2 * lg_floor(e - b));
        }
        __syncthreads();
        const int nbig = s_nbig;
        if (nbig > 0) {
            // s_ex and s_ofs are free until the next level: s_mark over s_ex, the pair
            // positions over s_ofs.  Group ends are marked before any piece start, so a piece
            // starting where another group ends keeps its mark.
            for (int i = t; i <= n; i += kBfsThreads) s_mark[i] = kMarkNone;
            __syncthreads();
            for (int g = t; g < nbig; g += kBfsThreads) s_mark[s_big[g].y] = kMarkGroupEnd;
            for (int g = 0; g < nbig; ++g) {
                __syncthreads();
                const int2 gr = s_big[g];
                mark_group<NW>(s_packed, gr.x, gr.y, 2 * lg_floor(gr.y - gr.x), s_mark, s_ofs,
                               s_ofs + kBfsCap / 2, s_part, s_lnext);
            }
            __syncthreads();
            wave_pieces<NW>(s_packed, n, s_mark, s_ofs, s_ofs + kBfsCap / 2, s_lnext);
            finish_pieces(s_packed, 0, n, s_mark);
        }
        __syncthreads();
        for (int i = t; i < n; i += kBfsThreads) {
            const int w = (int)(uint32_t)s_packed[i];
            s_front[i] = w;
            walk[base + i] = w;
            seq[w] = base + i;
        }
        base += n;
        f = n;
        ++level;
    }
    if (t == 0) *state = make_int4(f, base, level, overrun ? kBfsOverrun : finished ? 1 : 0);
}

// ---- 4b. a level of any size, four kernels over its edges ----------------------------------
// Work-groups own contiguous runs of frontier vertices (level_run), waves eight of them at a time:
// the wave's lanes go over the eight adjacency lists end to end (WaveEdges), so short lists share a
// round.  An edge's place among its work-group's edges is then also its children's order: (parent,
// ascending id).
// In a graph with a vertex of more than kHubDegree neighbours (HUBS) the lists are cut into segments
// of kSegment edges first, two more kernels a level, and the waves take eight segments at a time: the
// order of segments is the order of edges.  With a hub's list on one wave, ordering four hubs joined
// to 1 M vertices each took 72.6 ms, now 5.1 (20 kernels a level, as below, 23.5); 20 hubs of 0.1 M
// neighbours 26.9, now 5.4; R-MAT scale 18 4.3, now 2.4.
// With sizes known to the host a level took ~20 kernels (a radix sort of (parent, id) keys, scans,
// sorts of the groups) and four host round trips: the ordering of a 27-point mesh 64^3 in random
// numbering, 53 levels above 8192 edges, 14.3 -> 3.6 ms, its relabelling included.
constexpr int kLevelBlocks = 1024, kLevelWaves = 4, kLevelVerts = 8;
constexpr int kLevelStage = 512;  // children a wave sorts in LDS at a time
constexpr int kHubDegree = 2048, kSegment = 512;

// Counters of a level: {child groups left to k_level_sort, pieces of the split ones, segments,
// ranges left by every split pass}.
enum : int { kGroups, kPieces, kSegments, kRanges };
constexpr int kSplitPasses = 24;
constexpr int kCounters = kRanges + kSplitPasses;

// A segment: the place of its vertex, its first edge and edges, and -1, or (of a vertex cut into
// several) 4 times its job, plus kFirstSegment and kLastSegment.
enum : int { kFirstSegment = 1, kLastSegment = 2 };

__device__ __forceinline__ bool level_over(const int4& s, long long max_level) {
    return s.w || s.x == 0 || s.z > max_level;
}

// The frontier vertices [x, y) of this work-group.
__device__ __forceinline__ int2 level_run(int f) {
    constexpr int step = kLevelWaves * kLevelVerts;
    const int per = ((f + kLevelBlocks - 1) / kLevelBlocks + step - 1) / step * step;
    const long long b = (long long)blockIdx.x * per;
    return make_int2((int)min(b, (long long)f), (int)min(b + per, (long long)f));
}

// The edges of frontier items v0 .. v1 - 1 (at most kLevelVerts vertices, or HUBS: segments), end to
// end.  Lanes past the last item hold excl = total, so vertex() never picks them for e < total; of
// equal excl the last holds the edge, the lists before it being empty.
template <bool HUBS>
struct WaveEdges {
    int begin, excl, total;  // lane i < 8: its item's list, and the edges before it
    int place, part;         // lane i < 8: its vertex's place, its segment's last word
    __device__ __forceinline__ WaveEdges(const int* walk, const int* head, const int4* segs, int at,
                                         int v0, int v1) {
        const int lane = threadIdx.x & 63;
        int deg = 0;
        begin = 0;
        place = at + v0 + lane;
        part = -1;
        if (v0 + lane < v1) {
            if constexpr (HUBS) {
                const int4 g = segs[v0 + lane];
                place = g.x;
                begin = g.y;
                deg = g.z;
                part = g.w;
            } else {
                const int v = walk[place];
                begin = head[v];
                deg = head[v + 1] - begin;
            }
        }
        const int incl = wave_scan(deg, OpAdd{}, 0);
        excl = incl - deg;
        total = wave_last(incl);
    }
    // The place of item v's vertex: every lane together.
    __device__ __forceinline__ int parent(int v) const {
        if constexpr (HUBS) return __shfl(place, v);
        else return place - (int)(threadIdx.x & 63) + v;
    }
    // The item (0 .. 7) of edge e < total, and the edge's index in adj: every lane together.
    __device__ __forceinline__ int vertex(int e, int& index) const {
        int v = 0;
#pragma unroll
        for (int step = kLevelVerts / 2; step > 0; step >>= 1)
            if (__shfl(excl, v + step) <= e) v += step;
        index = __shfl(begin, v) + e - __shfl(excl, v);
        return v;
    }
    // f(neighbour, item, also's value, whether the lane holds an edge) for 64 edges at a time, in
    // order, all lanes together.  The loop waits for memory: U rounds' neighbours, and what `also`
    // loads for each, are in flight at once (eight rounds where the lists are long).
    template <int U, typename Also, typename F>
    __device__ __forceinline__ void rounds(const int* adj, Also&& also, F&& f) const {
        const int lane = threadIdx.x & 63;
        for (int e0 = 0; e0 < total; e0 += 64 * U) {
            int u[U], v[U], x[U];
#pragma unroll
            for (int q = 0; q < U; ++q) {
                int index;
                v[q] = vertex(min(e0 + 64 * q + lane, total - 1), index);
                u[q] = adj[index];
            }
#pragma unroll
            for (int q = 0; q < U; ++q) x[q] = also(u[q]);
#pragma unroll
            for (int q = 0; q < U; ++q)
                if (e0 + 64 * q < total) f(u[q], v[q], x[q], e0 + 64 * q + lane < total);
        }
    }
    template <typename Also, typename F>
    __device__ __forceinline__ void each(const int* adj, Also&& also, F&& f) const {
        if (total <= 512) rounds<4>(adj, also, f);
        else rounds<8>(adj, also, f);
    }
};

// Segments of each work-group's run of frontier vertices.
__global__ __launch_bounds__(256) void k_level_seg_count(
    const int* __restrict__ walk, const int* __restrict__ head, const int4* __restrict__ state,
    long long max_level, int* __restrict__ block_segs, int* __restrict__ counters) {
    __shared__ int total;
    const int4 s = *state;
    if (blockIdx.x == 0 && threadIdx.x < kCounters) counters[threadIdx.x] = 0;
    if (level_over(s, max_level)) return;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    const int2 run = level_run(s.x);
    int n = 0;
    for (int i = run.x + (int)threadIdx.x; i < run.y; i += 256) {
        const int v = walk[s.y - s.x + i];
        n += (head[v + 1] - head[v] + kSegment - 1) / kSegment;
    }
    n = wave_last(wave_scan(n, OpAdd{}, 0));
    if ((threadIdx.x & 63) == 0 && n) atomicAdd(&total, n);
    __syncthreads();
    if (threadIdx.x == 0) block_segs[blockIdx.x] = total;
}

// The sums of `counts` over the work-groups before this one and over all, by 256 threads.
__device__ __forceinline__ void block_sums(const int* __restrict__ counts, int& before, int& all,
                                           int* part /* LDS[2] */) {
    if (threadIdx.x < 2) part[threadIdx.x] = 0;
    __syncthreads();
    int b = 0, a = 0;
    for (int i = threadIdx.x; i < kLevelBlocks; i += 256) {
        const int c = counts[i];
        a += c;
        if (i < (int)blockIdx.x) b += c;
    }
    b = wave_last(wave_scan(b, OpAdd{}, 0));
    a = wave_last(wave_scan(a, OpAdd{}, 0));
    if ((threadIdx.x & 63) == 0) {
        atomicAdd(&part[0], b);
        atomicAdd(&part[1], a);
    }
    __syncthreads();
    before = part[0];
    all = part[1];
}

// The segments, in order.  A vertex of several gets a job of its own here; k_level_place fills in
// where its children begin and end.
__global__ __launch_bounds__(256) void k_level_seg_write(
    const int* __restrict__ walk, const int* __restrict__ head, const int4* __restrict__ state,
    long long max_level, const int* __restrict__ block_segs, int4* __restrict__ segs,
    int4* __restrict__ jobs, int* __restrict__ counters) {
    __shared__ int part[2], wsum[4];
    const int4 s = *state;
    if (level_over(s, max_level)) return;
    int out, all;
    block_sums(block_segs, out, all, part);
    if (blockIdx.x == 0 && threadIdx.x == 0) counters[kSegments] = all;
    const int2 run = level_run(s.x);
    for (int i0 = run.x; i0 < run.y; i0 += 256) {
        const int i = i0 + (int)threadIdx.x, place = s.y - s.x + i;
        int begin = 0, deg = 0;
        if (i < run.y) {
            const int v = walk[place];
            begin = head[v];
            deg = head[v + 1] - begin;
        }
        const int n = (deg + kSegment - 1) / kSegment;
        int sum;
        const int at = out + block_scan_256(n, OpAdd{}, 0, wsum, sum) - n;
        if (n == 1) segs[at] = make_int4(place, begin, deg, -1);
        if (n > 1) {
            const int job = atomicAdd(&counters[kGroups], 1);
            jobs[job] = make_int4(0, 0, -1, 0);
            for (int k = 0; k < n; ++k)
                segs[at + k] =
                    make_int4(place, begin + k * kSegment, min(kSegment, deg - k * kSegment),
                              4 * job + (k == 0 ? kFirstSegment : 0) + (k == n - 1 ? kLastSegment : 0));
        }
        out += sum;
        __syncthreads();
    }
}

template <bool HUBS>
__global__ __launch_bounds__(64 * kLevelWaves) void k_level_claim(
    const int* __restrict__ walk, const int* __restrict__ head, const int* __restrict__ adj,
    const int4* __restrict__ segs, const int* __restrict__ seq, int* claim,
    const int4* __restrict__ state, long long max_level, int* __restrict__ counters) {
    const int4 s = *state;
    if (!HUBS && blockIdx.x == 0 && threadIdx.x < kCounters) counters[threadIdx.x] = 0;
    if (level_over(s, max_level)) return;
    const int2 run = level_run(HUBS ? counters[kSegments] : s.x);
    const int at = s.y - s.x, w = threadIdx.x >> 6;
    for (int v0 = run.x + w * kLevelVerts; v0 < run.y; v0 += kLevelWaves * kLevelVerts) {
        const WaveEdges<HUBS> E(walk, head, segs, at, v0, min(v0 + kLevelVerts, run.y));
        E.each(adj, [&](int u) { return seq[u]; },
               [&](int u, int v, int placed, bool edge) {
                   const int parent = E.parent(v);
                   if (edge && placed < 0) atomicMin(&claim[u], parent);
               });
    }
}

// Children of each work-group's run.
template <bool HUBS>
__global__ __launch_bounds__(64 * kLevelWaves) void k_level_count(
    const int* __restrict__ walk, const int* __restrict__ head, const int* __restrict__ adj,
    const int4* __restrict__ segs, const int* __restrict__ claim, const int4* __restrict__ state,
    long long max_level, int* __restrict__ block_children, const int* __restrict__ counters) {
    __shared__ int total;
    const int4 s = *state;
    if (level_over(s, max_level)) return;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    const int2 run = level_run(HUBS ? counters[kSegments] : s.x);
    const int at = s.y - s.x, w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int n = 0;
    for (int v0 = run.x + w * kLevelVerts; v0 < run.y; v0 += kLevelWaves * kLevelVerts) {
        const WaveEdges<HUBS> E(walk, head, segs, at, v0, min(v0 + kLevelVerts, run.y));
        E.each(adj, [&](int u) { return claim[u]; },
               [&](int, int v, int parent, bool edge) {
                   const bool mine = parent == E.parent(v) && edge;
                   n += __popcll(__ballot(mine));
               });
    }
    if (lane == 0 && n) atomicAdd(&total, n);
    __syncthreads();
    if (threadIdx.x == 0) block_children[blockIdx.x] = total;
}

// Places the children: packed degree << 32 | id in child[], in (parent, ascending id) order.  A
// wave's children are staged in LDS, where each vertex's are sorted by one lane, and take their
// places; vertices with more than kBfsSortSmall children, and all of a wave with more than
// kLevelStage, become jobs {begin, end, partition depth} for k_level_sort, as those of several
// segments are already (depth -1: from the size).  The next state goes to `next`.
template <bool HUBS>
__global__ __launch_bounds__(64 * kLevelWaves) void k_level_place(
    int* walk, const int* __restrict__ head, const int* __restrict__ adj,
    const int4* __restrict__ segs, int* seq, const int* __restrict__ claim,
    const int4* __restrict__ state, int4* __restrict__ next, long long max_level,
    const int* __restrict__ block_children, u64* __restrict__ child, int4* __restrict__ jobs,
    int* __restrict__ counters) {
    __shared__ u64 s_stage[kLevelWaves][kLevelStage];
    __shared__ int s_cnt[kLevelWaves][kLevelVerts];
    __shared__ int s_round[2][kLevelWaves];
    __shared__ int s_part[2];
    const int4 s = *state;
    if (level_over(s, max_level)) {
        if (blockIdx.x == 0 && threadIdx.x == 0) *next = make_int4(s.x, s.y, s.z, s.w | (s.x == 0));
        return;
    }
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    int out, all, phase = 0;  // out: children before this round's items
    block_sums(block_children, out, all, s_part);
    if (blockIdx.x == 0 && t == 0) *next = make_int4(all, s.y + all, s.z + 1, all == 0);
    const int2 run = level_run(HUBS ? counters[kSegments] : s.x);
    const int at = s.y - s.x;
    const u64 below = lane ? (~0ull >> (64 - lane)) : 0ull;
    for (int r0 = run.x; r0 < run.y; r0 += kLevelWaves * kLevelVerts, phase ^= 1) {
        const int v0 = min(r0 + w * kLevelVerts, run.y), v1 = min(v0 + kLevelVerts, run.y);
        const WaveEdges<HUBS> E(walk, head, segs, at, v0, v1);
        if (lane < kLevelVerts) s_cnt[w][lane] = 0;
        wave_lds_fence();
        // the wave's children, staged as far as they fit
        int n = 0;
        E.each(adj, [&](int u) { return claim[u]; },
               [&](int u, int v, int parent, bool edge) {
                   const bool mine = parent == E.parent(v) && edge;
                   const u64 m = __ballot(mine);
                   if (mine) {
                       atomicAdd(&s_cnt[w][v], 1);
                       const int p = n + __popcll(m & below);
                       if (p < kLevelStage)
                           s_stage[w][p] =
                               (u64)(uint32_t)(head[u + 1] - head[u]) << 32 | (uint32_t)u;
                   }
                   n += __popcll(m);
               });
        if (lane == 0) s_round[phase][w] = n;
        __syncthreads();
        int mine_at = out, round = 0;
        for (int x = 0; x < kLevelWaves; ++x) {
            if (x < w) mine_at += s_round[phase][x];
            round += s_round[phase][x];
        }
        out += round;
        const int cnt = lane < kLevelVerts ? s_cnt[w][lane] : 0;
        const int first = wave_scan(cnt, OpAdd{}, 0) - cnt;  // lane i < 8: its children's start
        const bool part = HUBS && E.part >= 0;  // of a vertex that has its job
        if (part) {
            int* const job = reinterpret_cast<int*>(jobs + (E.part >> 2));
            if (E.part & kFirstSegment) job[0] = mine_at + first;
            if (E.part & kLastSegment) job[1] = mine_at + first + cnt;
        }
        const bool sorts = !part && cnt > (n <= kLevelStage ? kBfsSortSmall : 0);
        if (sorts)
            jobs[atomicAdd(&counters[kGroups], 1)] =
                make_int4(mine_at + first, mine_at + first + cnt, 2 * lg_floor(cnt), 0);
        if (n <= kLevelStage) {
            if (!part && !sorts && cnt > 1)
                ls_sort_range(s_stage[w], first, first + cnt, 2 * lg_floor(cnt));
            wave_lds_fence();
            for (int p0 = 0; p0 < n; p0 += 64) {
                const int p = p0 + lane;
                // the item of child p: is its group a job?
                int v = 0;
#pragma unroll
                for (int step = kLevelVerts / 2; step > 0; step >>= 1)
                    if (__shfl(first, v + step) <= min(p, n - 1)) v += step;
                const bool job = __shfl((int)(part || sorts), v);
                if (p < n) {
                    const u64 c = s_stage[w][p];
                    if (job) {
                        child[mine_at + p] = c;
                    } else {
                        const int u = (int)(uint32_t)c;
                        walk[s.y + mine_at + p] = u;
                        seq[u] = s.y + mine_at + p;
                    }
                }
            }
        } else {
            int k = 0;
            E.each(adj, [&](int u) { return claim[u]; },
                   [&](int u, int v, int parent, bool edge) {
                       const bool mine = parent == E.parent(v) && edge;
                       const u64 m = __ballot(mine);
                       if (mine)
                           child[mine_at + k + __popcll(m & below)] =
                               (u64)(uint32_t)(head[u + 1] - head[u]) << 32 | (uint32_t)u;
                       k += __popcll(m);
                   });
        }
        wave_lds_fence();
    }
}

// Partition depth of a job or range: the library's for its size where it is not known yet.
__device__ __forceinline__ int job_depth(const int4& job) {
    return job.z < 0 ? 2 * lg_floor(max(job.y - job.x, 1)) : job.z;
}

// A range of a group is done with once it fits k_level_sort, or its depth is used up: a piece, which
// joins the jobs after the groups.
__device__ __forceinline__ bool range_done(int lo, int hi, int depth) {
    return hi - lo <= kBfsCap || depth == 0;
}

__device__ __forceinline__ void add_piece(int4* jobs, int* counters, int lo, int hi, int depth) {
    jobs[counters[kGroups] + atomicAdd(&counters[kPieces], 1)] = make_int4(lo, hi, depth, 0);
}

// Groups of more than kBfsCap children: one partition step of every range, a work-group each, in
// memory (lpos, rpos at the range's own places).  The ranges of pass 0 are the jobs; what is not done
// with goes to the next pass.  One work-group from start to end took 9.3 ms for 1 M children of equal
// degree, parts side by side take 3.
__global__ __launch_bounds__(kBfsThreads) void k_level_split_pass(
    const int4* src, int pass, int4* __restrict__ dst, int4* jobs, int* counters, u64* child,
    int* lpos, int* rpos) {
    constexpr int NW = kBfsThreads / 64;
    __shared__ int2 s_part[NW];
    __shared__ int s_lnext;
    const int n = pass == 0 ? counters[kGroups] : counters[kRanges + pass - 1];
    for (int q = blockIdx.x; q < n; q += gridDim.x) {
        const int4 job = src[q];
        if (job.y - job.x <= kBfsCap) continue;
        __syncthreads();
        const int depth = job_depth(job) - 1;
        const int cut = partition_step<NW>(child, job.x, job.y, lpos + job.x, rpos + job.x, s_part,
                                           &s_lnext);
        if (threadIdx.x < 2) {
            const int lo = threadIdx.x ? cut : job.x, hi = threadIdx.x ? job.y : cut;
            if (range_done(lo, hi, depth)) add_piece(jobs, counters, lo, hi, depth);
            else dst[atomicAdd(&counters[kRanges + pass], 1)] = make_int4(lo, hi, depth, 0);
        }
    }
}

// The ranges that the passes left (parts of unlike sizes), each to its end in one work-group.
__global__ __launch_bounds__(kBfsThreads) void k_level_split(const int4* __restrict__ src, int passes,
                                                             int4* jobs, int* counters, u64* child,
                                                             int* lpos, int* rpos) {
    constexpr int NW = kBfsThreads / 64;
    __shared__ int2 s_part[NW];
    __shared__ int s_lnext;
    const int n = counters[kRanges + passes - 1];
    for (int q = blockIdx.x; q < n; q += gridDim.x) {
        const int4 job = src[q];
        __syncthreads();
        partition_range<NW>(child, job.x, job.y, job.z, kBfsCap, lpos + job.x, rpos + job.x,
                            s_part, &s_lnext, [&](int x, int y, int d) {
                                if (threadIdx.x == 0) add_piece(jobs, counters, x, y, d);
                            });
    }
}

// The groups k_level_place left, and the pieces of those that were split: one work-group each,
// in LDS; a piece beyond it has its depth used up and is heapsorted.
__global__ __launch_bounds__(kBfsThreads) void k_level_sort(
    const int4* __restrict__ jobs, const int* __restrict__ counters,
    const int4* __restrict__ state, u64* child, int* __restrict__ walk, int* __restrict__ seq) {
    constexpr int NW = kBfsThreads / 64;
    __shared__ u64 s_child[kBfsCap];
    __shared__ int s_lpos[kBfsCap / 2], s_rpos[kBfsCap / 2];
    __shared__ unsigned char s_mark[kBfsCap + 4];
    __shared__ int2 s_part[NW];
    __shared__ int s_lnext[NW];
    const int t = threadIdx.x, groups = counters[kGroups], all = groups + counters[kPieces];
    const int base = state->y;  // vertices placed before this level
    for (int q = blockIdx.x; q < all; q += gridDim.x) {
        const int4 job = jobs[q];
        const int n = job.y - job.x;
        u64* a = s_child;
        __syncthreads();
        if (n <= kBfsCap) {
            for (int i = t; i < n; i += kBfsThreads) {
                s_child[i] = child[job.x + i];
                s_mark[i] = kMarkNone;
            }
            __syncthreads();
            mark_group<NW>(s_child, 0, n, job_depth(job), s_mark, s_lpos, s_rpos, s_part, s_lnext);
            __syncthreads();
            wave_pieces<NW>(s_child, n, s_mark, s_lpos, s_rpos, s_lnext);
            finish_pieces(s_child, 0, n, s_mark);
        } else {
            if (q < groups) continue;  // its pieces follow
            a = child + job.x;
            if (t == 0) ls_heapsort(a, 0, n);
        }
        __syncthreads();
        for (int i = t; i < n; i += kBfsThreads) {
            const int u = (int)(uint32_t)a[i];
            walk[base + job.x + i] = u;
            seq[u] = base + job.x + i;
        }
    }
}

// ---- 5. order ----------------------------------------------------------------------------
// The component of place i's vertex: its root's place, roots being placed in rank order.
__global__ void k_order_keys(const int* __restrict__ walk, const int* __restrict__ comp,
                             const int* __restrict__ seq, int N, uint32_t* __restrict__ key) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) key[i] = (uint32_t)seq[comp[walk[i]]];
}

__global__ void k_positions(const uint32_t* __restrict__ order, int N, int* __restrict__ position) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) position[order[i]] = N - 1 - (int)i;
}

// ---- relabelling -------------------------------------------------------------------------
__global__ void k_perm_check(const int* __restrict__ position, int N, int* __restrict__ seen,
                             int* __restrict__ err) {
    const long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= N) return;
    const int p = position[v];
    if (p < 0 || p >= N || atomicAdd(&seen[p], 1) != 0) atomicOr(err, kBadPerm);
}

__global__ void k_relabel_keys(const int* __restrict__ row_of, const int* __restrict__ col,
                               const int* __restrict__ position, long long nnz, int nb,
                               u64* __restrict__ key, uint32_t* __restrict__ val) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nnz) return;
    key[p] = (u64)row_of[p] << nb | (u64)position[col[p]];
    val[p] = (uint32_t)p;
}

// Two equal sorted (row, new column) keys: a row holds a column twice.  Checked before
// anything is written, so a rejected call leaves the caller's CSR as it was.
__global__ void k_relabel_dups(const u64* __restrict__ key, long long nnz,
                               int* __restrict__ err) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i > 0 && i < nnz && key[i - 1] == key[i]) atomicOr(err, kDupCol);
}

__global__ void k_relabel_gather(const u64* __restrict__ key, const uint32_t* __restrict__ src,
                                 const float* __restrict__ vin, long long nnz, int nb,
                                 int* __restrict__ cout, float* __restrict__ vout) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnz) return;
    cout[i] = (int)(key[i] & ((1ull << nb) - 1));
    vout[i] = vin[src[i]];
}

// Rows relabelled and sorted by new column on their own, since they do not move: up to 64
// nonzeros by one wave, each lane counting the row's columns below its own; longer ones, up to
// kRowSortMax, are listed and sorted by a work-group in LDS (bitonic).  A radix sort of (row, column)
// keys of the whole matrix, which rows beyond that still take, moved 12 bytes a nonzero five times.
// 27-point mesh 64^3, 6.9 M nonzeros: 95 us, ordering and relabelling 14.3 -> 13.8 ms.
// A wave a row costs 0.19 ns a row, nonzeros or not, the keys about 0.09 ns a nonzero and 0.1 ms for
// their launches: many rows of fewer than two nonzeros on average take the keys.  Rows alone / keys,
// us, the checks included: 1 M rows of 0.3 M nonzeros 284 / 307, of 1 M 336 / 332, of 4 M 385 / 502;
// 10 M rows of 1 M 1365 / 392, of 10 M 2100 / 968; 50 M rows of 1 M 3790 / 556; 3 M rows of 30 M
// 1226 / 2690.
constexpr int kRowsAlone = 1 << 20;  // up to this many rows never take the keys for being short
constexpr int kRowSortMax = 4096;

// One atomic a work-group, of which a launch has at most kLongestBlocks: one a wave took 17 ns a wave
// (relabelling 10 M rows of 1 M nonzeros 2.7 -> 1.4 ms).
constexpr unsigned kLongestBlocks = 1024;

__global__ __launch_bounds__(256) void k_longest_row(const int* __restrict__ rp, int M,
                                                     int* __restrict__ longest) {
    __shared__ int most;
    if (threadIdx.x == 0) most = 0;
    __syncthreads();
    int m = 0;
    for (long long r = (long long)blockIdx.x * 256 + threadIdx.x; r < M; r += 256ll * gridDim.x)
        m = max(m, rp[r + 1] - rp[r]);
    m = wave_last(wave_scan(m, OpMax{}, 0));
    if ((threadIdx.x & 63) == 0) atomicMax(&most, m);
    __syncthreads();
    if (threadIdx.x == 0 && most > 0) atomicMax(longest, most);
}

__global__ __launch_bounds__(256) void k_relabel_rows(
    const int* __restrict__ rp, const int* __restrict__ col, const float* __restrict__ val,
    const int* __restrict__ position, int M, int* __restrict__ cout, float* __restrict__ vout,
    int* __restrict__ listed, int* __restrict__ nlisted, int* __restrict__ err) {
    const long long r = group_index() * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    if (r >= M) return;  // the whole wave
    const int a = __builtin_amdgcn_readfirstlane(rp[r]);
    const int len = __builtin_amdgcn_readfirstlane(rp[r + 1]) - a;
    if (len > 64) {
        if (lane == 0) listed[atomicAdd(nlisted, 1)] = (int)r;
        return;
    }
    int c = INT_MAX;
    float v = 0.0f;
    if (lane < len) {
        c = position[col[a + lane]];
        v = val[a + lane];
    }
    int rank = 0, same = 0;
    for (int i = 0; i < len; ++i) {
        const int x = __builtin_amdgcn_readlane(c, i);
        rank += x < c;
        same += x == c;
    }
    if (lane < len) {
        if (same > 1) atomicOr(err, kDupCol);  // nothing of this is kept then
        cout[a + rank] = c;
        vout[a + rank] = v;
    }
}

__global__ __launch_bounds__(256) void k_relabel_listed(
    const int* __restrict__ rp, const int* __restrict__ col, const float* __restrict__ val,
    const int* __restrict__ position, const int* __restrict__ listed,
    const int* __restrict__ nlisted, int* __restrict__ cout, float* __restrict__ vout,
    int* __restrict__ err) {
    __shared__ u64 key[kRowSortMax];  // new column << 32 | index in the row
    const int t = threadIdx.x, n = *nlisted;
    for (int q = blockIdx.x; q < n; q += gridDim.x) {
        const int r = listed[q], a = rp[r], len = rp[r + 1] - a;
        int size = 128;
        while (size < len) size *= 2;
        __syncthreads();
        for (int i = t; i < size; i += 256)
            key[i] = i < len ? (u64)(uint32_t)position[col[a + i]] << 32 | (uint32_t)i : ~0ull;
        for (int k = 2; k <= size; k *= 2)
            for (int j = k / 2; j > 0; j /= 2) {
                __syncthreads();
                for (int p = t; p < size / 2; p += 256) {
                    const int i = 2 * p - (p & (j - 1)), o = i + j;
                    const u64 x = key[i], y = key[o];
                    if ((x > y) == ((i & k) == 0)) {
                        key[i] = y;
                        key[o] = x;
                    }
                }
            }
        __syncthreads();
        for (int i = t; i < len; i += 256) {
            const u64 x = key[i];
            if (i > 0 && (uint32_t)(key[i - 1] >> 32) == (uint32_t)(x >> 32))
                atomicOr(err, kDupCol);
            cout[a + i] = (int)(x >> 32);
            vout[a + i] = val[a + (int)(uint32_t)x];
        }
    }
}

// B_out[position[r], :] = B[r, :]; one thread per V consecutive floats of a row of W * V.
template <int V>
__global__ void k_permute_rows(const float* __restrict__ B, const int* __restrict__ position,
                               long long n, unsigned W, float* __restrict__ Bout) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    long long r;
    if (n <= 0xffffffffll) r = (unsigned)i / W;
    else r = i / W;
    const long long k = i - r * W;
    reinterpret_cast<vec*>(Bout)[(long long)position[r] * W + k] =
        reinterpret_cast<const vec*>(B)[i];
}

__global__ void k_mark_heads(const int* __restrict__ rp, int M, int* __restrict__ head) {
    const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= M) return;
    const int a = rp[r];
    if (a < rp[r + 1]) head[a] = (int)r;
}

// Row of every nonzero: each non-empty row marks its first slot, a running max fills the rest.
void row_of_nonzeros(const int* rp, int M, int nnz, int* row_of, hipStream_t st) {
    TmpBuf<int> headmark(nnz);
    fill<int>(headmark.p, nnz, (int)0x80000000, st);
    RLAUNCH(k_mark_heads, M, rp, M, headmark.p);
    inclusive_max(headmark.p, row_of, nnz, st);
}

// The distinct (vertex, neighbour) pairs in order; returns their number.
template <typename K>
long long adjacency(const int* rp, const int* col, int M, int N, int nnz, int nb,
                    TmpBuf<int>& adj_u, TmpBuf<int>& adj, hipStream_t st) {
    const long long P = 2ll * nnz;
    if (P == 0) return 0;
    TmpBuf<int> row_of(nnz);
    row_of_nonzeros(rp, M, nnz, row_of.p, st);
    TmpBuf<K> k1(P), k2(P);
    RLAUNCH((k_adj_pairs<K>), nnz, row_of.p, col, (long long)nnz, N, nb, k1.p);
    row_of.release();
    K *ka = k1.p, *kb = k2.p;
    radix_sort_keys<K>(ka, kb, P, 2 * nb, st);
    TmpBuf<int> flag(P), pos(P + 1);
    RLAUNCH((k_unique_flags<K>), P, ka, P, flag.p);
    exclusive_sum<int, int>(flag.p, pos.p, P, st);
    const long long E = read_scalar(pos.p + P, st);
    adj_u.alloc(E);
    adj.alloc(E);
    RLAUNCH((k_unique_write<K>), P, ka, pos.p, P, nb, adj_u.p, adj.p);
    return E;
}

// Iteration limits of the ordering's loops; 0 selects the proven maxima (see rcm_order_device).
// Process-wide, read once by each ordering.
std::atomic<long long> g_max_level{0}, g_max_rounds{0};

}  // namespace

void set_rcm_limits(long long max_level, long long max_rounds) {
    g_max_level.store(max_level, std::memory_order_relaxed);
    g_max_rounds.store(max_rounds, std::memory_order_relaxed);
}

void rcm_order_device(const int* rp, const int* col, int M, int N, int nnz, int* position,
                      hipStream_t st) {
    if (M < 0 || N < 0 || nnz < 0) throw Error(VCSRMC_ERR_ARG, "negative matrix size");
    if (!rp || (nnz > 0 && !col) || (N > 0 && !position))
        throw Error(VCSRMC_ERR_ARG, "null pointer");
    if (2ll * nnz >= (1ll << 31))
        throw Error(VCSRMC_ERR_OVERFLOW, "rcm ordering handles fewer than 2^30 nonzeros");
    ScratchScope scratch((size_t)(72ll * nnz + 160ll * N));
    TmpBuf<int> err(1);
    check_csr(rp, col, M, N, nnz, err.p, st);
    if (N == 0) return;

    const int nb = std::max(1, bits_for((u64)N));  // holds 0..N
    // 1. adjacency
    TmpBuf<int> adj_u, adj, head((size_t)N + 1);
    const long long E = 2 * nb <= 32
                            ? adjacency<uint32_t>(rp, col, M, N, nnz, nb, adj_u, adj, st)
                            : adjacency<u64>(rp, col, M, N, nnz, nb, adj_u, adj, st);
    key_ptr<int>(adj_u.p, E, N, head.p, st);

    // 2. rank
    TmpBuf<uint32_t> k1(N), k2(N), v1(N), v2(N);
    uint32_t *ka = k1.p, *kb = k2.p, *va = v1.p, *vb = v2.p;
    TmpBuf<int> rank(N);
    RLAUNCH(k_rank_keys, N, head.p, N, ka, va);
    radix_sort_pairs<uint32_t>(ka, va, kb, vb, N, nb, st);  // a degree is at most N
    const uint32_t* order = va;
    const int max_degree = (int)read_scalar(ka + (N - 1), st);
    RLAUNCH(k_scatter_rank, N, order, N, rank.p);

    // Proven maxima of the loops below.  Levels: every level but the last places at least one
    // vertex, so level <= N.  Component rounds: a round changes something or ends the loop;
    // between two rounds with a hook (each hook removes a tree, so at most N - 1 of them),
    // pointer jumping alone halves every depth, so after ceil(lg N) + 1 rounds all trees are
    // stars and the next round either hooks or changes nothing: at most
    // N (ceil(lg N) + 2) + 1 rounds.
    const long long lim_level = g_max_level.load(std::memory_order_relaxed);
    const long long lim_rounds = g_max_rounds.load(std::memory_order_relaxed);
    const long long max_level = lim_level > 0 ? lim_level : (long long)N + 1;
    const long long max_rounds =
        lim_rounds > 0 ? lim_rounds : (long long)N * (bits_for((u64)N) + 2) + 1;

    // 3. components.  Rounds are enqueued a few at a time, each with its own flag; rounds after
    // one that changed nothing change nothing either.
    TmpBuf<int> comp(N);
    {
        constexpr int kBatch = 4;
        TmpBuf<int> changed(kBatch);
        RLAUNCH(k_cc_init, N, comp.p, N);
        for (long long round = 0;;) {
            if (round >= max_rounds)
                throw Error(VCSRMC_ERR_STATE, "rcm ordering: connected components did not settle "
                                              "within " + std::to_string(max_rounds) + " rounds");
            const int batch = (int)std::min<long long>(kBatch, max_rounds - round);
            fill<int>(changed.p, kBatch, 0, st);
            for (int i = 0; i < batch; ++i) {
                RLAUNCH(k_cc_hook, E, adj_u.p, adj.p, E, rank.p, comp.p, changed.p + i);
                RLAUNCH(k_cc_jump, N, comp.p, N, changed.p + i);
            }
            int flags[kBatch];
            VCSRMC_HIP(hipMemcpyAsync(flags, changed.p, sizeof flags, hipMemcpyDeviceToHost, st));
            VCSRMC_HIP(hipStreamSynchronize(st));
            if (std::find(flags, flags + batch, 0) != flags + batch) break;
            round += batch;
        }
    }
    adj_u.release();

    // 4. levels
    TmpBuf<int> seq(N), claim(N), walk(N);
    fill<int>(seq.p, N, -1, st);
    fill<int>(claim.p, N, INT_MAX, st);
    TmpBuf<int4> state(2);
    int roots = 0;
    {
        TmpBuf<int> flag(N), pos((size_t)N + 1);
        RLAUNCH(k_root_flags, N, order, comp.p, N, flag.p);
        exclusive_sum<int, int>(flag.p, pos.p, N, st);
        roots = read_scalar(pos.p + N, st);
        RLAUNCH(k_root_list, N, order, flag.p, pos.p, N, walk.p, seq.p);
    }
    TmpBuf<u64> child(N);
    // A group or piece holds at least one child and there are at most N of each.  Without a vertex
    // of more than kBfsSortSmall neighbours no group becomes a job (nor do eight fill more than
    // kLevelStage), and none needs splitting without one of more than kBfsCap.
    static_assert(kLevelVerts * kBfsSortSmall <= kLevelStage, "small groups always fit");
    static_assert(kHubDegree >= kBfsSortSmall, "segments need the jobs");
    const bool sorts = max_degree > kBfsSortSmall, splits = max_degree > kBfsCap;
    const bool hubs = max_degree > kHubDegree;
    TmpBuf<int4> jobs(sorts ? 2 * (size_t)N : 0);
    TmpBuf<int> counters(kCounters), lpos(splits ? N : 0), rpos(splits ? N : 0);
    TmpBuf<int> children(kLevelBlocks), block_segs(hubs ? kLevelBlocks : 0);
    // every vertex ends at most one segment that is not full
    TmpBuf<int4> segs(hubs ? (size_t)N + (size_t)(E / kSegment) : 0);
    // Passes that halve the largest possible group down to kBfsCap, and one more; ranges above it
    // number at most N / kBfsCap.
    const int passes = splits ? std::min(bits_for((u64)(max_degree / kBfsCap)) + 1, kSplitPasses) : 0;
    TmpBuf<int4> ranges0(splits ? N / kBfsCap + 1 : 0), ranges1(splits ? N / kBfsCap + 1 : 0);
    int4 s = make_int4(roots, roots, 1, 0);
    VCSRMC_HIP(hipMemcpyAsync(state.p, &s, sizeof s, hipMemcpyHostToDevice, st));
    int cur = 0;
    const dim3 grid(kLevelBlocks), block(64 * kLevelWaves);
    const auto level = [&](auto with_hubs, const int4* now, int4* next) {
        constexpr bool HUBS = decltype(with_hubs)::value;
        if constexpr (HUBS) {
            hipLaunchKernelGGL(k_level_seg_count, grid, dim3(256), 0, st, walk.p, head.p, now,
                               max_level, block_segs.p, counters.p);
            VCSRMC_HIP(hipGetLastError());
            hipLaunchKernelGGL(k_level_seg_write, grid, dim3(256), 0, st, walk.p, head.p, now,
                               max_level, block_segs.p, segs.p, jobs.p, counters.p);
            VCSRMC_HIP(hipGetLastError());
        }
        hipLaunchKernelGGL((k_level_claim<HUBS>), grid, block, 0, st, walk.p, head.p, adj.p, segs.p,
                           seq.p, claim.p, now, max_level, counters.p);
        VCSRMC_HIP(hipGetLastError());
        hipLaunchKernelGGL((k_level_count<HUBS>), grid, block, 0, st, walk.p, head.p, adj.p, segs.p,
                           claim.p, now, max_level, children.p, counters.p);
        VCSRMC_HIP(hipGetLastError());
        hipLaunchKernelGGL((k_level_place<HUBS>), grid, block, 0, st, walk.p, head.p, adj.p, segs.p,
                           seq.p, claim.p, now, next, max_level, children.p, child.p, jobs.p,
                           counters.p);
        VCSRMC_HIP(hipGetLastError());
    };
    for (int batch = 1; s.y < N && !s.w && s.z <= max_level; batch = std::min(2 * batch, 16)) {
        // levels inside one work-group while they are small, then `batch` of any size
        hipLaunchKernelGGL(k_bfs_levels, dim3(1), dim3(kBfsThreads), 0, st, walk.p, head.p, adj.p,
                           seq.p, claim.p, N, max_level, state.p + cur);
        VCSRMC_HIP(hipGetLastError());
        for (int i = 0; i < batch; ++i, cur ^= 1) {
            const int4* now = state.p + cur;
            if (hubs) level(std::true_type{}, now, state.p + (cur ^ 1));
            else level(std::false_type{}, now, state.p + (cur ^ 1));
            const int4* src = jobs.p;
            for (int pass = 0; pass < passes; ++pass) {
                int4* dst = pass % 2 ? ranges1.p : ranges0.p;
                hipLaunchKernelGGL(k_level_split_pass, dim3(256), dim3(kBfsThreads), 0, st, src, pass,
                                   dst, jobs.p, counters.p, child.p, lpos.p, rpos.p);
                VCSRMC_HIP(hipGetLastError());
                src = dst;
            }
            if (splits) {
                hipLaunchKernelGGL(k_level_split, dim3(256), dim3(kBfsThreads), 0, st, src, passes,
                                   jobs.p, counters.p, child.p, lpos.p, rpos.p);
                VCSRMC_HIP(hipGetLastError());
            }
            if (sorts) {
                hipLaunchKernelGGL(k_level_sort, dim3(256), dim3(kBfsThreads), 0, st, jobs.p,
                                   counters.p, now, child.p, walk.p, seq.p);
                VCSRMC_HIP(hipGetLastError());
            }
        }
        s = read_scalar(state.p + cur, st);
    }
    if (s.y != N) {
        if (s.w == kBfsOverrun || s.z > max_level)
            throw Error(VCSRMC_ERR_STATE, "rcm ordering: the breadth-first walk passed " +
                                              std::to_string(max_level) + " levels");
        throw Error(VCSRMC_ERR_STATE, "rcm ordering left vertices unvisited");
    }

    // 5. order: the walk, its components one after another
    const uint32_t* last = reinterpret_cast<const uint32_t*>(walk.p);
    if (roots > 1) {
        RLAUNCH(k_order_keys, N, walk.p, comp.p, seq.p, N, k1.p);
        last = radix_sort_pairs_from<uint32_t>(k1.p, last, k2.p, v1.p, k1.p, v2.p, N,
                                               bits_for((u64)(roots - 1)), st).second;
    }
    RLAUNCH(k_positions, N, last, N, position);
    VCSRMC_HIP(hipStreamSynchronize(st));
    scratch.idle();
}

void apply_column_permutation_device(const int* rp, int* col, float* val, int M, int N, int nnz,
                                     const int* position, const float* B, int O, float* B_out,
                                     hipStream_t st) {
    if (M < 0 || N < 0 || nnz < 0 || O < 0) throw Error(VCSRMC_ERR_ARG, "negative size");
    if (!rp || (nnz > 0 && (!col || !val)) || (N > 0 && !position))
        throw Error(VCSRMC_ERR_ARG, "null pointer");
    if ((B == nullptr) != (B_out == nullptr))
        throw Error(VCSRMC_ERR_ARG, "B and B_out must both be given or both be NULL");
    if (B && B == B_out) throw Error(VCSRMC_ERR_ARG, "B_out must not alias B");
    // rows on their own: columns and values; else keys and payloads too (rows beyond kRowSortMax,
    // which are not known yet, ask for those when they come to it)
    const bool rows_alone = M <= kRowsAlone || 2ll * M <= nnz;
    ScratchScope scratch((size_t)((rows_alone ? 8ll : 36ll) * nnz + 8ll * N + 4ll * M));
    // every check of the input at once: {errors, longest row}
    TmpBuf<int> err(2), seen(N);
    fill<int>(err.p, 2, 0, st);
    RLAUNCH(k_check_rp, (long long)M + 1, rp, M, nnz, err.p);
    if (M > 0) {
        hipLaunchKernelGGL(k_longest_row, dim3(std::min(nblk(M), kLongestBlocks)), dim3(256), 0, st,
                           rp, M, err.p + 1);
        VCSRMC_HIP(hipGetLastError());
    }
    RLAUNCH(k_check_cols, (long long)nnz, col, (long long)nnz, N, err.p);
    fill<int>(seen.p, N, 0, st);
    RLAUNCH(k_perm_check, N, position, N, seen.p, err.p);
    raise_if(err.p, st);
    if (nnz > 0) {
        const int longest = read_scalar(err.p + 1, st);
        TmpBuf<int> ncol(nnz);
        TmpBuf<float> nval(nnz);
        if (longest <= kRowSortMax && rows_alone) {
            TmpBuf<int> listed(longest > 64 ? M : 0), nlisted(1);
            fill<int>(nlisted.p, 1, 0, st);
            hipLaunchKernelGGL(k_relabel_rows, grid_of(((long long)M + 3) / 4), dim3(256), 0, st, rp,
                               col, val, position, M, ncol.p, nval.p, listed.p, nlisted.p, err.p);
            VCSRMC_HIP(hipGetLastError());
            if (longest > 64) {
                hipLaunchKernelGGL(k_relabel_listed, dim3(2048), dim3(256), 0, st, rp, col, val,
                                   position, listed.p, nlisted.p, ncol.p, nval.p, err.p);
                VCSRMC_HIP(hipGetLastError());
            }
        } else {
            const int nb = std::max(1, bits_for((u64)N));
            const int mb = std::max(1, bits_for((u64)M));
            TmpBuf<int> row_of(nnz);
            row_of_nonzeros(rp, M, nnz, row_of.p, st);
            TmpBuf<u64> k1(nnz), k2(nnz);
            TmpBuf<uint32_t> v1(nnz), v2(nnz);
            RLAUNCH(k_relabel_keys, nnz, row_of.p, col, position, (long long)nnz, nb, k1.p, v1.p);
            row_of.release();
            u64 *ka = k1.p, *kb = k2.p;
            uint32_t *va = v1.p, *vb = v2.p;
            radix_sort_pairs<u64>(ka, va, kb, vb, nnz, nb + mb, st);
            RLAUNCH(k_relabel_dups, nnz, ka, (long long)nnz, err.p);
            RLAUNCH(k_relabel_gather, nnz, ka, va, val, (long long)nnz, nb, ncol.p, nval.p);
        }
        raise_if(err.p, st);
        VCSRMC_HIP(hipMemcpyAsync(col, ncol.p, sizeof(int) * (size_t)nnz, hipMemcpyDeviceToDevice,
                                  st));
        VCSRMC_HIP(hipMemcpyAsync(val, nval.p, sizeof(float) * (size_t)nnz,
                                  hipMemcpyDeviceToDevice, st));
    }
    if (B && N > 0 && O > 0) {
        const bool wide = O % 4 == 0 && ((uintptr_t)B | (uintptr_t)B_out) % 16 == 0;
        const long long n = wide ? (long long)N * (O / 4) : (long long)N * O;
        if (wide) RLAUNCH((k_permute_rows<4>), n, B, position, n, (unsigned)(O / 4), B_out);
        else RLAUNCH((k_permute_rows<1>), n, B, position, n, (unsigned)O, B_out);
    }
    VCSRMC_HIP(hipStreamSynchronize(st));
    scratch.idle();
}

}  // namespace vcsrmc
