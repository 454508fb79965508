// row_groups.hip -- a row order for the execution layout that puts rows sharing columns into the
// same 16-row panel.
//
// A panel's tiles are its distinct columns, 32 at a time, so a panel of rows that share columns
// has fewer tiles: fewer matrix-core steps, fewer B rows gathered, fuller tiles.  Natural order
// is often far from that: a 27-point stencil on a grid in natural order puts 16 consecutive x
// positions in a panel (a 16 x 1 x 1 strip, 162 distinct columns, 6 tiles), where a 4 x 2 x 2
// block of the same rows touches 96 (3 tiles).
//
// Method: multilevel heavy-edge matching on the row-column incidence.  Level k pairs clusters of
// up to 2^k rows, so four levels give groups of up to 16.  At each level every cluster scores
// the clusters it shares columns with (columns of more than `hub` rows are ignored: they link
// rows without telling them apart), keeps its best few, and clusters whose first choices are
// each other merge; a few rounds let clusters whose partner was taken try their next choice.
// The score is the number of shared columns; ties go to the pair whose first rows r < s satisfy
// floor(r / (s - r)) even, then to the nearer pair (the farther at the last level), then to a
// hash of the pair.  The parity rule makes chains of equally good partners pair up in phase
// (rows 0-1, 2-3, ... rather than a pairing that shifts from one chain to the next), which is
// what lets the next level merge the pairs into compact blocks; the distance rule keeps pairs
// near in the original order, except at the last level, where the farther of equally good
// partners makes a panel span more of the slowest direction of the natural order (z of a 3D
// grid: 2 x 2 x 4 blocks of a 27-point stencil, not 4 x 2 x 2; the same 96 columns): the B
// rows of a z-plane, reused by the panels one plane away long after one XCD's L2 has dropped
// them, are then fetched by 1.5 slabs of panels instead of 2.  Measured on gfx950 (kernel us,
// C += A.B / C = A.B): 27-point 100^3 FP32 444 / 347 -> 424 / 343, FP16 306 / 233 -> 308 /
// 225; 7-point 100^3 FP32 367 / 254 -> 354 / 253, FP16 268 / 194 -> 272 / 185; 7-point 60^3
// FP32 65.7 / 53.6 -> 60.7 / 48.1, FP16 48.3 / 29.8 -> 45.9 / 31.5; 2D 5-point grids unchanged.
// Finally the rows are ordered by their group's first row (rows in a group by index); rows
// without nonzeros go last, so they fill no panel.
//
// Every loop is bounded (levels, rounds, probes, insertions per cluster: a cluster whose
// candidates overflow its table keeps the ones it counted first), and the sorts are stable.
#include <algorithm>
#include <climits>
#include <tuple>

#include "internal.hpp"
#include "primitives.hpp"

namespace vcsrmc {
namespace {

typedef unsigned long long u64;

constexpr int kLevels = 4;            // 2^4 = kPanelRows rows per group
constexpr int kRounds = 8;            // proposal rounds per level
constexpr int kCand = 4;              // candidates kept per cluster and level
constexpr int kTableBits = 10;
constexpr int kTable = 1 << kTableBits;  // LDS hash table slots per wave (one cluster)
constexpr int kProbes = 64;           // linear probes per insertion
constexpr int kMaxCols = 512;         // clusters with more (non-hub) columns take no partner
constexpr int kInsertsPerLane = 256;  // candidate insertions per lane and cluster

inline unsigned grid256(long long n) { return grid_for(n, 256); }
inline dim3 waves_of(long long n) { return grid_of((n + 3) / 4); }  // four in a work-group

__device__ __forceinline__ unsigned mix32(unsigned x) {
    x ^= x >> 16;
    x *= 0x7feb352du;
    x ^= x >> 15;
    x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The largest of 64 values (and each lane's own value back): DPP scans, no LDS.
__device__ __forceinline__ u64 wave_max_u64(u64 x) {
    const int hi = (int)(unsigned)(x >> 32);  // below 2^31 (the count has 13 bits)
    const int top = __builtin_amdgcn_readlane(wave_scan(hi, OpMax{}, INT_MIN), 63);
    const int lo = hi == top ? (int)((unsigned)x ^ 0x80000000u) : INT_MIN;
    const int low = __builtin_amdgcn_readlane(wave_scan(lo, OpMax{}, INT_MIN), 63);
    return ((u64)(unsigned)top << 32) | ((unsigned)low ^ 0x80000000u);
}

__global__ void k_any_hub(const int* __restrict__ cptr, int N, int hub, int* __restrict__ any) {
    const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (c < N && cptr[c + 1] - cptr[c] > hub) *any = 1;
}

// The entries whose column is not a hub.
__global__ void k_keep_flags(const int* __restrict__ col, const int* __restrict__ cptr,
                             long long n, int hub, int* __restrict__ keep) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int c = col[i];
    keep[i] = cptr[c + 1] - cptr[c] <= hub;
}

__global__ void k_keep_write(const int* __restrict__ row_of, const int* __restrict__ col,
                             const int* __restrict__ keep, const int* __restrict__ at, long long n,
                             uint32_t* __restrict__ kcol, uint32_t* __restrict__ krow) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && keep[i]) {
        kcol[at[i]] = (uint32_t)col[i];
        krow[at[i]] = (uint32_t)row_of[i];
    }
}

// ptr[v] = entries before row v that were kept (rp[v] of them existed).
__global__ void k_keep_ptr(const int* __restrict__ rp, const int* __restrict__ at, int M,
                           int* __restrict__ ptr) {
    const long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v <= M) ptr[v] = at[rp[v]];
}

// One wave per cluster a: counts, in an LDS hash table, how many of a's columns each other
// cluster b holds, then keeps the kCand best b with size(a) + size(b) <= maxsz (see the file
// comment for the order).  cand[a * kCand + i] = b, or -1.
// Issue slots bound it: a 27-point stencil inserts 27 x 27 candidates a row and finds 125
// clusters.  So a column's list is shared by as many lanes as its cluster's columns leave idle,
// its entries are loaded four at a time ahead of the insertions, and the table is squeezed to its
// filled slots before any of them is scored.  Scoring all 1024 slots, a lane a column and an
// entry at a time, the four levels of the stencil 100^3 took 10.9 ms; now 4.4.
__global__ __launch_bounds__(256) void k_score(const uint32_t* __restrict__ ccol,
                                               const int* __restrict__ cr_ptr,
                                               const uint32_t* __restrict__ rcl,
                                               const int* __restrict__ rc_ptr,
                                               const int* __restrict__ size,
                                               const int* __restrict__ cmin, int nc, int maxsz,
                                               bool far, int4* __restrict__ cand) {
    __shared__ __attribute__((aligned(16))) int tkey[4][kTable];
    __shared__ __attribute__((aligned(16))) int tcnt[4][kTable];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long long wa = group_index() * 4 + w;
    if (wa >= nc) return;  // the whole wave
    const int a = __builtin_amdgcn_readfirstlane((int)wa);
    int* K = tkey[w];
    int* Cn = tcnt[w];
    const int b0 = cr_ptr[a], b1 = cr_ptr[a + 1];
    const int sa = size[a];
    const int ncol = b1 - b0;
    static_assert(kCand == 4, "candidates are stored as one int4");
    if (ncol > kMaxCols || ncol == 0 || sa >= maxsz) {
        if (lane == 0) cand[a] = make_int4(-1, -1, -1, -1);
        return;
    }
    for (int i = lane * 4; i < kTable; i += 256) {
        *reinterpret_cast<int4*>(K + i) = make_int4(-1, -1, -1, -1);
        *reinterpret_cast<int4*>(Cn + i) = make_int4(0, 0, 0, 0);
    }
    wave_sync();
    int sh = 0;  // 2^sh lanes share a column
    while ((ncol << (sh + 1)) <= 64) ++sh;
    const int S = 1 << sh;
    int inserted = 0;
    for (int ci = b0 + (lane >> sh); ci < b1 && inserted < kInsertsPerLane; ci += 64 >> sh) {
        const int c = (int)ccol[ci];
        const int r1 = rc_ptr[c + 1];
        for (int j = rc_ptr[c] + (lane & (S - 1)); j < r1 && inserted < kInsertsPerLane;
             j += 4 * S) {
            int b[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) b[q] = j + q * S < r1 ? (int)rcl[j + q * S] : a;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (b[q] == a) continue;
                ++inserted;
                unsigned h = ((unsigned)b[q] * 0x9e3779b1u) >> (32 - kTableBits);
                for (int p = 0; p < kProbes; ++p) {
                    const int prev = atomicCAS(&K[h], -1, b[q]);
                    if (prev == -1 || prev == b[q]) {
                        atomicAdd(&Cn[h], 1);
                        break;
                    }
                    h = (h + 1) & (kTable - 1);
                }
            }
        }
    }
    wave_sync();
    // The filled slots, in slot order, to the table's front: slot group s goes to places at or
    // before its own, which have been read.
    int nd = 0;
    const u64 below = lane ? (~0ull >> (64 - lane)) : 0ull;
    for (int s = 0; s < kTable / 64; ++s) {
        const int k = K[lane + 64 * s], n = Cn[lane + 64 * s];
        const u64 filled = __ballot(k >= 0);
        wave_sync();
        if (k >= 0) {
            const int at = nd + __popcll(filled & below);
            K[at] = k;
            Cn[at] = n;
        }
        nd += __popcll(filled);
        wave_sync();
    }
    // Score keys: shared columns, phase, nearness, hash; each lane keeps its kCand best.
    u64 best[kCand];
    int who[kCand];
#pragma unroll
    for (int i = 0; i < kCand; ++i) {
        best[i] = 0;
        who[i] = -1;
    }
    const int ma = cmin[a];
    for (int e = lane; e < nd; e += 64) {
        int b = K[e];
        if (sa + size[b] > maxsz) continue;
        const int mb = cmin[b];
        const int lo = min(ma, mb), d = max(ma, mb) - lo;  // d >= 1: distinct first rows
        const u64 cnt = (u64)min(Cn[e], 8191);
        const u64 phase = ((lo / d) & 1) == 0;
        const u64 near = far ? (u64)d : (u64)(0x7fffffff - d);
        const u64 tie =
            mix32((unsigned)min(a, b) * 0x9e3779b9u ^ (unsigned)max(a, b)) & 0x3ffffu;
        u64 key = (cnt << 50) | (phase << 49) | (near << 18) | tie;
#pragma unroll
        for (int i = 0; i < kCand; ++i) {
            const bool up = key > best[i];
            const u64 k = up ? best[i] : key;
            const int x = up ? who[i] : b;
            best[i] = up ? key : best[i];
            who[i] = up ? b : who[i];
            key = k;
            b = x;
        }
    }
    // kCand rounds of a wave-wide maximum; the lanes holding it move to their next.  Keys of two
    // candidates tie only if their nearness, phase and 18-bit pair hash all agree, and then the
    // lowest lane's candidate is kept and the other dropped.
    int out[kCand];
#pragma unroll
    for (int r = 0; r < kCand; ++r) {
        const u64 top = wave_max_u64(best[0]);
        const u64 own = __ballot(best[0] == top);
        out[r] = top ? __builtin_amdgcn_readlane(who[0], (int)__builtin_ctzll(own)) : -1;
        if (best[0] == top) {
#pragma unroll
            for (int i = 0; i + 1 < kCand; ++i) {
                best[i] = best[i + 1];
                who[i] = who[i + 1];
            }
            best[kCand - 1] = 0;
        }
    }
    if (lane == 0) cand[a] = make_int4(out[0], out[1], out[2], out[3]);
}

// A cluster still unmatched proposes to its first candidate that is unmatched too.
__global__ void k_propose(const int* __restrict__ cand, const int* __restrict__ mate, int nc,
                          int* __restrict__ prop) {
    const long long a = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= nc) return;
    int p = -1;
    if (mate[a] < 0) {
        for (int i = 0; i < kCand; ++i) {
            const int b = cand[a * kCand + i];
            if (b >= 0 && mate[b] < 0) {
                p = b;
                break;
            }
        }
    }
    prop[a] = p;
}

// Mutual proposals match (each side records its own partner).
__global__ void k_accept(const int* __restrict__ prop, int nc, int* __restrict__ mate) {
    const long long a = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= nc) return;
    const int b = prop[a];
    if (b >= 0 && prop[b] == (int)a) mate[a] = b;
}

// The merged cluster keeps the id rank of its smaller member.
__global__ void k_rep_flags(const int* __restrict__ mate, int nc, int* __restrict__ isrep) {
    const long long a = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (a < nc) isrep[a] = mate[a] < 0 || (int)a < mate[a];
}

__global__ void k_relabel(const int* __restrict__ mate, const int* __restrict__ nid,
                          const int* __restrict__ size, const int* __restrict__ cmin, int nc,
                          int* __restrict__ newcl, int* __restrict__ nsize,
                          int* __restrict__ ncmin, int2* __restrict__ parts) {
    const long long a = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= nc) return;
    const int m = mate[a];
    const int rep = (m >= 0 && m < (int)a) ? m : (int)a;
    newcl[a] = nid[rep];
    if (rep == (int)a) {
        nsize[nid[a]] = size[a] + (m >= 0 ? size[m] : 0);
        ncmin[nid[a]] = m >= 0 ? min(cmin[a], cmin[m]) : cmin[a];
        parts[nid[a]] = make_int2((int)a, m);
    }
}

__global__ void k_relabel_rows(const int* __restrict__ newcl, int M, int* __restrict__ rowcl) {
    const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < M) rowcl[r] = newcl[rowcl[r]];
}

// Elements of the ascending v[lo, hi) below x.
__device__ __forceinline__ int below_in(const uint32_t* __restrict__ v, int lo, int hi,
                                        uint32_t x) {
    const int first = lo;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (v[mid] < x) lo = mid + 1;
        else hi = mid;
    }
    return lo - first;
}

// Column lists of the merged clusters, one wave each: the union of its parts' ascending lists, by
// rank (an element's place is its index plus the other list's elements before it, less the common
// ones before it), not by sorting all of them again.  k_union_sizes counts, k_union_write writes.
__global__ __launch_bounds__(256) void k_union_sizes(const int2* __restrict__ parts,
                                                     const int* __restrict__ ptr,
                                                     const uint32_t* __restrict__ ccol, int nnc,
                                                     int* __restrict__ len) {
    const long long wx = group_index() * 4 + (threadIdx.x >> 6);
    if (wx >= nnc) return;  // the whole wave
    const int x = (int)wx, lane = threadIdx.x & 63;
    const int2 p = parts[x];
    const int a0 = ptr[p.x], a1 = ptr[p.x + 1];
    int total = a1 - a0;
    if (p.y >= 0) {
        const int b0 = ptr[p.y], b1 = ptr[p.y + 1];
        total += b1 - b0;
        for (int j0 = b0; j0 < b1; j0 += 64) {
            bool common = false;
            if (j0 + lane < b1) {
                const uint32_t c = ccol[j0 + lane];
                const int at = a0 + below_in(ccol, a0, a1, c);
                common = at < a1 && ccol[at] == c;
            }
            total -= __popcll(__ballot(common));
        }
    }
    if (lane == 0) len[x] = total;
}

__global__ __launch_bounds__(256) void k_union_write(const int2* __restrict__ parts,
                                                     const int* __restrict__ ptr,
                                                     const uint32_t* __restrict__ ccol,
                                                     const int* __restrict__ nptr, int nnc,
                                                     uint32_t* __restrict__ ncol,
                                                     uint32_t* __restrict__ ncl) {
    const long long wx = group_index() * 4 + (threadIdx.x >> 6);
    if (wx >= nnc) return;  // the whole wave
    const int x = (int)wx, lane = threadIdx.x & 63;
    const u64 below = lane ? (~0ull >> (64 - lane)) : 0ull;
    const int2 p = parts[x];
    const int out = nptr[x];
#pragma unroll
    for (int side = 0; side < 2; ++side) {
        const int me = side ? p.y : p.x, other = side ? p.x : p.y;
        if (me < 0) break;
        const int a0 = ptr[me], a1 = ptr[me + 1];
        const int b0 = other >= 0 ? ptr[other] : 0, b1 = other >= 0 ? ptr[other + 1] : 0;
        int common_before = 0;
        for (int i0 = a0; i0 < a1; i0 += 64) {
            const int i = i0 + lane;
            bool common = false;
            int at = 0;
            uint32_t c = 0;
            if (i < a1) {
                c = ccol[i];
                at = below_in(ccol, b0, b1, c);
                common = b0 + at < b1 && ccol[b0 + at] == c;
            }
            const u64 m = __ballot(common);
            if (i < a1 && !(side && common)) {
                const int dst = out + (i - a0) + at - common_before - __popcll(m & below);
                ncol[dst] = c;
                ncl[dst] = (uint32_t)x;
            }
            common_before += __popcll(m);
        }
    }
}

__global__ void k_init_clusters(int M, int* __restrict__ rowcl, int* __restrict__ size,
                                int* __restrict__ cmin) {
    const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= M) return;
    rowcl[r] = (int)r;
    size[r] = 1;
    cmin[r] = (int)r;
}

// Order key of row r: its group's first row (rows without nonzeros last); the stable sort keeps
// the rows of a group by index.
__global__ void k_order_keys(const int* __restrict__ rowcl, const int* __restrict__ cmin,
                             const int* __restrict__ rp, int M,
                             uint32_t* __restrict__ key, uint32_t* __restrict__ pay) {
    const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= M) return;
    key[r] = rp[r + 1] > rp[r] ? (uint32_t)cmin[rowcl[r]] : (uint32_t)M;
    pay[r] = (uint32_t)r;
}

__global__ void k_positions(const uint32_t* __restrict__ order, int M, int P,
                            int* __restrict__ row_map) {
    const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p < P) row_map[p] = p < M ? (int)order[p] : -1;
}

__global__ void k_flag_rows(const int* __restrict__ rp, int M, int* __restrict__ flag) {
    const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r < M) flag[r] = rp[r + 1] > rp[r];
}

// Rows with nonzeros keep their order at positions 0..NE-1, the others follow in order.
__global__ void k_compact_positions(const int* __restrict__ flag, const int* __restrict__ rank,
                                    int M, int NE, int* __restrict__ row_map) {
    const long long r = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= M) return;
    const int p = flag[r] ? rank[r] : NE + ((int)r - rank[r]);
    row_map[p] = (int)r;
}

}  // namespace

bool compact_rows(const int* rp, int M, hipStream_t st, DevBuf<int>& row_map) {
    if (M < 1) return false;
    TmpBuf<int> flag(M), rank((size_t)M + 1);
    hipLaunchKernelGGL(k_flag_rows, dim3(grid256(M)), dim3(256), 0, st, rp, M, flag.p);
    VCSRMC_HIP(hipGetLastError());
    exclusive_sum<int, int>(flag.p, rank.p, M, st);
    const int NE = read_scalar(rank.p + M, st);
    if (8LL * (M - NE) < M) return false;
    const int P = ((M + kPanelRows - 1) / kPanelRows) * kPanelRows;
    row_map.alloc(P);
    fill<int>(row_map.p, P, -1, st);
    hipLaunchKernelGGL(k_compact_positions, dim3(grid256(M)), dim3(256), 0, st, flag.p, rank.p, M,
                       NE, row_map.p);
    VCSRMC_HIP(hipGetLastError());
    return true;
}

bool group_rows(const int* rp, const int* row_of, const int* col, long long n, int M, int N,
                hipStream_t st, DevBuf<int>& row_map) {
    if (M < 2 * kPanelRows || N < 1 || n < 1) return false;
    const int cbits = bits_for((unsigned long long)(N - 1));
    const int hub = (int)std::max<long long>(32, std::min<long long>(1024, 4 * n / N));

    // Level-0 clusters are the rows, without the columns of more than `hub` rows.  A cluster's
    // columns: cl_col (ascending) in [ptr[cluster], ptr[cluster + 1]), cl_of the cluster of each.
    TmpBuf<uint32_t> cl_col, cl_of;
    TmpBuf<int> cl_ptr;
    const uint32_t *ccol = reinterpret_cast<const uint32_t*>(col),
                   *cof = reinterpret_cast<const uint32_t*>(row_of);
    const int* ptr = rp;
    long long np = n;
    // column -> rows, ascending: the entries stably sorted by column.  The column lists of level 0
    // too: those of the columns it keeps are whole.  (Column degrees counted by atomics instead took
    // 25 ms with 8 columns of 1 M nonzeros.)
    TmpBuf<uint32_t> k1(n), k2(n), v1(n), v2(n);
    TmpBuf<int> rc_ptr((size_t)N + 1);
    const uint32_t *scol, *rcl;
    std::tie(scol, rcl) = radix_sort_pairs_from<uint32_t>(ccol, cof, k1.p, v1.p, k2.p, v2.p, n,
                                                          std::max(1, cbits), st);
    key_ptr<uint32_t>(scol, n, N, rc_ptr.p, st);
    {
        TmpBuf<int> any(1);
        fill<int>(any.p, 1, 0, st);
        hipLaunchKernelGGL(k_any_hub, dim3(grid256(N)), dim3(256), 0, st, rc_ptr.p, N, hub, any.p);
        VCSRMC_HIP(hipGetLastError());
        if (read_scalar(any.p, st)) {
            TmpBuf<int> keep(n), at((size_t)n + 1);
            hipLaunchKernelGGL(k_keep_flags, dim3(grid256(n)), dim3(256), 0, st, col, rc_ptr.p, n,
                               hub, keep.p);
            VCSRMC_HIP(hipGetLastError());
            exclusive_sum<int, int>(keep.p, at.p, n, st);
            np = read_scalar(at.p + n, st);
            if (np == 0) return false;
            cl_col.alloc(np);
            cl_of.alloc(np);
            cl_ptr.alloc((size_t)M + 1);
            hipLaunchKernelGGL(k_keep_write, dim3(grid256(n)), dim3(256), 0, st, row_of, col,
                               keep.p, at.p, n, cl_col.p, cl_of.p);
            VCSRMC_HIP(hipGetLastError());
            hipLaunchKernelGGL(k_keep_ptr, dim3(grid256((long long)M + 1)), dim3(256), 0, st, rp,
                               at.p, M, cl_ptr.p);
            VCSRMC_HIP(hipGetLastError());
            ccol = cl_col.p;
            cof = cl_of.p;
            ptr = cl_ptr.p;
        }
    }

    int nc = M;
    TmpBuf<int> rowcl(M), size(M), cmin(M);
    hipLaunchKernelGGL(k_init_clusters, dim3(grid256(M)), dim3(256), 0, st, M, rowcl.p, size.p,
                       cmin.p);
    VCSRMC_HIP(hipGetLastError());
    for (int level = 0; level < kLevels; ++level) {
        if (level > 0) {  // column -> clusters
            k1.alloc(np);
            k2.alloc(np);
            v1.alloc(np);
            v2.alloc(np);
            std::tie(scol, rcl) = radix_sort_pairs_from<uint32_t>(
                ccol, cof, k1.p, v1.p, k2.p, v2.p, np, std::max(1, cbits), st);
            key_ptr<uint32_t>(scol, np, N, rc_ptr.p, st);
        }

        const int maxsz = 2 << level;  // clusters of 2^level rows pair into 2^(level+1)
        TmpBuf<int4> cand(nc);
        TmpBuf<int> mate(nc), prop(nc);
        hipLaunchKernelGGL(k_score, waves_of(nc), dim3(256), 0, st, ccol, ptr, rcl,
                           rc_ptr.p, size.p, cmin.p, nc, maxsz, level == kLevels - 1, cand.p);
        VCSRMC_HIP(hipGetLastError());
        k1.release(); k2.release(); v1.release(); v2.release();
        fill<int>(mate.p, nc, -1, st);
        const int* candidates = reinterpret_cast<const int*>(cand.p);
        for (int round = 0; round < kRounds; ++round) {
            hipLaunchKernelGGL(k_propose, dim3(grid256(nc)), dim3(256), 0, st, candidates, mate.p,
                               nc, prop.p);
            VCSRMC_HIP(hipGetLastError());
            hipLaunchKernelGGL(k_accept, dim3(grid256(nc)), dim3(256), 0, st, prop.p, nc, mate.p);
            VCSRMC_HIP(hipGetLastError());
        }
        TmpBuf<int> isrep(nc), nid((size_t)nc + 1);
        hipLaunchKernelGGL(k_rep_flags, dim3(grid256(nc)), dim3(256), 0, st, mate.p, nc, isrep.p);
        VCSRMC_HIP(hipGetLastError());
        exclusive_sum<int, int>(isrep.p, nid.p, nc, st);
        const int nnc = read_scalar(nid.p + nc, st);
        if (nnc == nc) break;  // nothing merged at this level: none will at the next
        TmpBuf<int> newcl(nc), nsize(nnc), ncmin(nnc);
        TmpBuf<int2> parts(nnc);
        hipLaunchKernelGGL(k_relabel, dim3(grid256(nc)), dim3(256), 0, st, mate.p, nid.p, size.p,
                           cmin.p, nc, newcl.p, nsize.p, ncmin.p, parts.p);
        VCSRMC_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_relabel_rows, dim3(grid256(M)), dim3(256), 0, st, newcl.p, M,
                           rowcl.p);
        VCSRMC_HIP(hipGetLastError());
        size = std::move(nsize);
        cmin = std::move(ncmin);
        if (level + 1 < kLevels) {
            TmpBuf<int> len(nnc), nptr((size_t)nnc + 1);
            hipLaunchKernelGGL(k_union_sizes, waves_of(nnc), dim3(256), 0, st, parts.p,
                               ptr, ccol, nnc, len.p);
            VCSRMC_HIP(hipGetLastError());
            exclusive_sum<int, int>(len.p, nptr.p, nnc, st);
            const long long nu = read_scalar(nptr.p + nnc, st);
            TmpBuf<uint32_t> ncol(nu), ncl(nu);
            hipLaunchKernelGGL(k_union_write, waves_of(nnc), dim3(256), 0, st, parts.p,
                               ptr, ccol, nptr.p, nnc, ncol.p, ncl.p);
            VCSRMC_HIP(hipGetLastError());
            cl_col = std::move(ncol);
            cl_of = std::move(ncl);
            cl_ptr = std::move(nptr);
            ccol = cl_col.p;
            cof = cl_of.p;
            ptr = cl_ptr.p;
            np = nu;
        }
        nc = nnc;
    }

    // Rows by group (first row of the group), rows without nonzeros last.
    const int P = ((M + kPanelRows - 1) / kPanelRows) * kPanelRows;
    TmpBuf<uint32_t> okey(M), oalt(M), opay(M), opalt(M);
    hipLaunchKernelGGL(k_order_keys, dim3(grid256(M)), dim3(256), 0, st, rowcl.p, cmin.p, rp, M,
                       okey.p, opay.p);
    VCSRMC_HIP(hipGetLastError());
    uint32_t *ok = okey.p, *oka = oalt.p, *order = opay.p, *order_alt = opalt.p;
    radix_sort_pairs<uint32_t>(ok, order, oka, order_alt, M, bits_for((unsigned long long)M), st);
    row_map.alloc(P);
    hipLaunchKernelGGL(k_positions, dim3(grid256(P)), dim3(256), 0, st, order, M, P, row_map.p);
    VCSRMC_HIP(hipGetLastError());
    return true;
}

}  // namespace vcsrmc
