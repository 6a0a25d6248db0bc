// Neighbour-support (Verlet CSR) builder, device scan and transposed-CSR
// builder for gfx950.
//
// Support semantics follow the reference's Verlet list for DC-PSE
// (VL_NON_SYMMETRIC | VL_SKIP_REF_PART: q != p, |x_p - x_q| < rCut), see
// src/DCPSE/SupportBuilder.cuh:15-61. Unlike that builder (one thread per
// particle, host-side serial prefix sum, size_t keys, 4 host round trips), the
// whole CSR is built on the device: a cell grid by counting sort, then one
// wavefront per group of neighbouring particles (one set) or per particle over
// the neighbouring cells' particles, flattened into one candidate list and
// sorted in registers, so every row comes out in ascending particle index
// (deterministic, independent of atomic ordering).
#include <algorithm>
#include <climits>
#include <cmath>
#include <type_traits>

#include "dcpse_common.hpp"
#include "dcpse_internal.hpp"

namespace dcpse {

// ---------------------------------------------------------------------------
// scan
// ---------------------------------------------------------------------------
constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanBlock * kScanItems;

__global__ __launch_bounds__(kScanBlock) void k_scan_tilesum(const int32_t* __restrict__ in, int64_t n,
                                                             int64_t* __restrict__ tsum) {
    __shared__ long long red[kScanBlock / kWave];
    const int64_t base = (int64_t)blockIdx.x * kScanTile;
    long long s = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        int64_t k = base + (int64_t)i * kScanBlock + threadIdx.x;
        if (k < n) s += in[k];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, kWave);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        long long t = 0;
        for (int w = 0; w < kScanBlock / kWave; ++w) t += red[w];
        tsum[blockIdx.x] = t;
    }
}

// Exclusive scan of tsum[0..nt) in place, tsum[nt] = total. One block.
__global__ __launch_bounds__(1024) void k_scan_tilesums(int64_t* tsum, int64_t nt) {
    __shared__ long long buf[1024];
    long long carry = 0;
    for (int64_t b = 0; b < nt; b += 1024) {
        int64_t i = b + threadIdx.x;
        long long v = i < nt ? tsum[i] : 0;
        buf[threadIdx.x] = v;
        __syncthreads();
        for (int off = 1; off < 1024; off <<= 1) {
            long long t = threadIdx.x >= (unsigned)off ? buf[threadIdx.x - off] : 0;
            __syncthreads();
            buf[threadIdx.x] += t;
            __syncthreads();
        }
        if (i < nt) tsum[i] = carry + buf[threadIdx.x] - v;
        long long tot = buf[1023];
        __syncthreads();
        carry += tot;
    }
    if (threadIdx.x == 0) tsum[nt] = carry;
}

// Sum over the block of one value per thread, in every thread.
template <int BLOCK>
__device__ __forceinline__ long long block_sum(long long v) {
    __shared__ long long red[BLOCK / kWave];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    long long t = 0;
#pragma unroll
    for (int w = 0; w < BLOCK / kWave; ++w) t += red[w];
    __syncthreads();
    return t;
}

// One tile per block. tsum: the tiles' sums (scanned: their exclusive scan),
// or null where there is one tile.
template <int BLOCK>
__global__ __launch_bounds__(BLOCK) void k_scan_tiles(const int32_t* __restrict__ in, int64_t n,
                                                      const int64_t* __restrict__ tsum, bool scanned,
                                                      int64_t* __restrict__ out, int64_t* host,
                                                      const int32_t* extra0, const int32_t* extra1) {
    __shared__ long long wsum[BLOCK / kWave];
    const int64_t base = ((int64_t)blockIdx.x * BLOCK + threadIdx.x) * kScanItems;
    long long v[kScanItems];
    long long tot = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        int64_t k = base + i;
        v[i] = k < n ? in[k] : 0;
        tot += v[i];
    }
    long long before = 0;
    if (scanned) {
        before = tsum[blockIdx.x];
    } else if (tsum) {
        for (int64_t i = threadIdx.x; i < (int64_t)blockIdx.x; i += BLOCK) before += tsum[i];
        before = block_sum<BLOCK>(before);
    }
    // inclusive over the wavefront, then the wavefronts before this one
    long long incl = tot;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const long long t = __shfl_up(incl, off, kWave);
        if ((int)(threadIdx.x & 63) >= off) incl += t;
    }
    if ((threadIdx.x & 63) == 63) wsum[threadIdx.x >> 6] = incl;
    __syncthreads();
    long long all = before;
#pragma unroll
    for (int w = 0; w < BLOCK / kWave; ++w) {
        if (w < (int)(threadIdx.x >> 6)) before += wsum[w];
        all += wsum[w];
    }
    long long run = before + incl - tot;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        int64_t k = base + i;
        if (k < n) out[k] = run;
        run += v[i];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        out[n] = all;
        if (host) {
            host[0] = all;
            if (extra0) host[1] = *extra0;
            if (extra1) host[2] = *extra1;
            __threadfence_system();
        }
    }
}

__global__ void k_to_host(const int32_t* v, int64_t* host) {
    *host = *v;
    __threadfence_system();
}

size_t scan_workspace_bytes(int64_t n) {
    int64_t nt = (n + kScanTile - 1) / kScanTile;
    return (size_t)(nt + 1) * sizeof(int64_t) + 256;
}

dcpse_status scan_counts(dcpse_ctx* ctx, const int32_t* in, int64_t n, int64_t* out, Workspace* w, bool to_host,
                         const int32_t* extra0, const int32_t* extra1) {
    int64_t* host = to_host ? ctx->host : nullptr;
    // one launch up to a block of 1024 threads; then the tiles' sums first, each
    // block adding up those before its own (4.8 us a launch: lists of 2,500
    // particles ran six of these kernels, now two or three), scanned by a
    // kernel of their own where that would be long
    if (n <= 1024 * kScanItems) {
        k_scan_tiles<1024><<<1, 1024, 0, ctx->stream>>>(in, n, nullptr, false, out, host, extra0, extra1);
        DCPSE_LAUNCH_CHECK(ctx);
        return DCPSE_OK;
    }
    const int64_t nt = (n + kScanTile - 1) / kScanTile;
    int64_t* tsum = w->take<int64_t>((size_t)nt + 1);
    if (!tsum) return fail(ctx, DCPSE_ERR_INVALID, "scan: workspace too small");
    k_scan_tilesum<<<(unsigned)nt, kScanBlock, 0, ctx->stream>>>(in, n, tsum);
    DCPSE_LAUNCH_CHECK(ctx);
    const bool scanned = nt > 4096;
    if (scanned) {
        k_scan_tilesums<<<1, 1024, 0, ctx->stream>>>(tsum, nt);
        DCPSE_LAUNCH_CHECK(ctx);
    }
    k_scan_tiles<kScanBlock><<<(unsigned)nt, kScanBlock, 0, ctx->stream>>>(in, n, tsum, scanned, out, host, extra0,
                                                                          extra1);
    DCPSE_LAUNCH_CHECK(ctx);
    return DCPSE_OK;
}

__global__ void k_fill_i32(int32_t* p, int64_t n, int32_t v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

void fill_i32(hipStream_t s, int32_t* p, int64_t n, int32_t v) {
    if (n <= 0) return;
    int64_t blocks = std::min<int64_t>((n + 255) / 256, 65536);
    k_fill_i32<<<(unsigned)blocks, 256, 0, s>>>(p, n, v);
}

// Zeroes up to four ranges in one launch.
struct ClearRanges {
    int32_t* p[4];
    int64_t n[4];
};
__global__ void k_clear(const ClearRanges r) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
        for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < r.n[k]; i += (int64_t)gridDim.x * blockDim.x)
            r.p[k][i] = 0;
}

__global__ void k_fill_i64(int64_t* p, int64_t n, int64_t v) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

static void fill_i64(hipStream_t s, int64_t* p, int64_t n, int64_t v) {
    if (n <= 0) return;
    int64_t blocks = std::min<int64_t>((n + 255) / 256, 65536);
    k_fill_i64<<<(unsigned)blocks, 256, 0, s>>>(p, n, v);
}

bool captured(hipStream_t s) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (!s || hipStreamIsCapturing(s, &st) == hipSuccess) return st != hipStreamCaptureStatusNone;
    (void)hipGetLastError();
    return false;
}

WorkspaceUse::~WorkspaceUse() {
    if (captured(ctx->stream)) return;  // nothing runs before the graph is launched
    if (hipEventRecord(ctx->ws_event, ctx->stream) == hipSuccess) {
        ctx->ws_stream = ctx->stream;
        ctx->ws_queued = true;
    } else {  // no event to wait for later: wait now
        (void)hipGetLastError();
        (void)hipStreamSynchronize(ctx->stream);
    }
}

dcpse_status reserve_workspace(dcpse_ctx* ctx, size_t bytes, Workspace* w) {
    if (ctx->ws_queued && ctx->ws_stream != ctx->stream && !captured(ctx->stream))
        DCPSE_HIP_CHECK(ctx, hipStreamWaitEvent(ctx->stream, ctx->ws_event, 0));
    if (ctx->ws_size < bytes) {
        if (ctx->ws_queued) DCPSE_HIP_CHECK(ctx, hipEventSynchronize(ctx->ws_event));
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
        if (ctx->ws) DCPSE_HIP_CHECK(ctx, hipFree(ctx->ws));
        // nothing is left if the larger one cannot be had
        const size_t grown = std::max(bytes, ctx->ws_size * 2);
        ctx->ws = nullptr;
        ctx->ws_size = 0;
        for (size_t nb : {grown, bytes}) {
            const hipError_t e = hipMalloc(&ctx->ws, nb);
            if (e == hipSuccess) {
                ctx->ws_size = nb;
                break;
            }
            (void)hipGetLastError();  // not the next launch's error
            ctx->ws = nullptr;
            if (nb == bytes)
                return fail(ctx, DCPSE_ERR_HIP, "a workspace of %zu bytes: %s", bytes, hipGetErrorString(e));
        }
    }
    w->base = static_cast<char*>(ctx->ws);
    w->cap = ctx->ws_size;
    w->used = 0;
    return DCPSE_OK;
}

// ---------------------------------------------------------------------------
// cell grid
// ---------------------------------------------------------------------------
struct CellGrid {
    int nc[3];
    int kmax[3];  // cells scanned on each side: ceil(largest rcut / cs), capped so a periodic wrap visits no cell twice
    double lo[3], cs[3], len[3], ilen[3];
    unsigned periodic;
    int64_t ncell;
};

__device__ __forceinline__ int cell_of(double x, int d, const CellGrid& g) {
    double t = floor((x - g.lo[d]) / g.cs[d]);
    t = fmin(fmax(t, -1.0e9), 1.0e9);
    int v = (int)t;
    if ((g.periodic >> d) & 1u) {
        v %= g.nc[d];
        if (v < 0) v += g.nc[d];
    } else {
        v = min(max(v, 0), g.nc[d] - 1);
    }
    return v;
}

// A particle in cell order: position and index side by side, so that a
// candidate is one 32-byte access, in the scattered write as in the reads
// (a 1.89M-particle list: assignment and fill 115 us, 205 us with separate
// arrays and a second atomic pass).
struct __align__(16) CellRec {
    double x[3];
    int32_t id;
    int32_t pad;
};

template <int DIM>
__device__ __forceinline__ int32_t cell_index(const double* x, const CellGrid& g) {
    int64_t c = 0, stride = 1;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        c += stride * cell_of(x[d], d, g);
        stride *= g.nc[d];
    }
    return (int32_t)c;
}

// Home groups of a set with a cut-off per particle: level l holds the
// particles whose cut-off lies in (rtop / 2^(l+1), rtop / 2^l] (the last level
// all smaller ones) on a grid of its own, of edge about kHomeEdge times the
// level's largest cut-off; first[l] is the level's first cell in one numbering.
// An edge of 0.85 cut-offs puts 8 to 70 particles into a group at 58
// neighbours each: enough to share the candidates' setup, few enough that most
// candidates are some particle's neighbours.
constexpr int kMaxLevels = 6;
constexpr double kHomeEdge = 0.85;
struct HomeLevels {
    int n;
    double rtop;
    CellGrid g[kMaxLevels];
    int32_t first[kMaxLevels + 1];
};

// cnt[c] += 1, returning the place taken: lanes side by side with the same c
// (particles next to each other in memory mostly share a cell) take theirs with
// one atomic. Called by the first `active` lanes of the wavefront.
__device__ __forceinline__ int32_t take_place(int32_t* cnt, int32_t c, int active) {
    const int lane = threadIdx.x & 63;
    const int prev = __shfl_up(c, 1, kWave);
    const bool head = lane == 0 || prev != c;
    const unsigned long long heads = __ballot(head);
    const unsigned long long upto = (2ull << lane) - 1;
    const int first = 63 - __builtin_clzll(heads & upto);
    const unsigned long long after = heads & ~upto;
    const int end = after ? __builtin_ctzll(after) : active;
    int32_t base = 0;
    if (head) base = atomicAdd(&cnt[c], end - lane);
    return __shfl(base, first, kWave) + lane - first;
}

// cell of every particle and its place within it (the order within a cell is
// whatever the atomics give; nothing that leaves the builder depends on it).
template <int DIM, bool HOME>
__global__ void k_cell_assign(const double* __restrict__ pos, int64_t n, const double* __restrict__ rcut, CellGrid g,
                              HomeLevels h, int32_t* __restrict__ cell_id, int32_t* __restrict__ rank,
                              int32_t* __restrict__ cell_cnt, int32_t* __restrict__ home_id,
                              int32_t* __restrict__ home_rank, int32_t* __restrict__ home_cnt) {
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n;
         q += (int64_t)gridDim.x * blockDim.x) {
        double x[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) x[d] = pos[d * n + q];
        const int32_t c = cell_index<DIM>(x, g);
        cell_id[q] = c;
        const int active = (int)min((int64_t)kWave, n - (q - (threadIdx.x & 63)));
        rank[q] = take_place(cell_cnt, c, active);
        if constexpr (HOME) {
            const double r = rcut[q];
            int l = 0;
            double below = 0.5 * h.rtop;
            while (l + 1 < h.n && r <= below) {
                ++l;
                below *= 0.5;
            }
            int32_t k = 0;
#pragma unroll
            for (int i = 0; i < kMaxLevels; ++i)
                if (i == l) k = h.first[i] + cell_index<DIM>(x, h.g[i]);
            home_id[q] = k;
            home_rank[q] = take_place(home_cnt, k, active);
        }
    }
}

// The records of the particles in cell order (and in home order).
template <int DIM, bool HOME>
__global__ void k_cell_fill(const double* __restrict__ pos, int64_t n, const int32_t* __restrict__ cell_id,
                            const int32_t* __restrict__ rank, const int64_t* __restrict__ cell_start,
                            CellRec* __restrict__ rec, const int32_t* __restrict__ home_id,
                            const int32_t* __restrict__ home_rank, const int64_t* __restrict__ home_start,
                            CellRec* __restrict__ home_rec) {
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n;
         q += (int64_t)gridDim.x * blockDim.x) {
        CellRec r;
        r.x[2] = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) r.x[d] = pos[d * n + q];
        r.id = (int32_t)q;
        r.pad = 0;
        rec[cell_start[cell_id[q]] + rank[q]] = r;
        if constexpr (HOME) home_rec[home_start[home_id[q]] + home_rank[q]] = r;
    }
}

// flag[i] = whether cell i holds a particle
__global__ void k_occupied(const int32_t* __restrict__ cnt, int64_t n, int32_t* __restrict__ flag) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        flag[i] = cnt[i] > 0;
}

// The occupied cells in order: group_cell[index[i]] = i (index: exclusive scan
// of the flags).
__global__ void k_group_cells(const int32_t* __restrict__ cnt, const int64_t* __restrict__ index, int64_t n,
                              int32_t* __restrict__ group_cell) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        if (cnt[i] > 0) group_cell[index[i]] = (int32_t)i;
}

constexpr int kRowWaves = 4;  // wavefronts per block in the row kernels

// v of lane ^ S (S a power of two below 64): DPP within quads and rows,
// ds_swizzle within 32-lane halves, ds_bpermute across them.
template <int S>
__device__ __forceinline__ int lane_xor(int v, int lane) {
    if constexpr (S == 1) return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);   // quad_perm 1,0,3,2
    else if constexpr (S == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);  // quad_perm 2,3,0,1
    else if constexpr (S == 8) return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, false);  // row_ror 8
    else if constexpr (S == 4 || S == 16) return __builtin_amdgcn_ds_swizzle(v, 0x1F | (S << 10));  // and 31, xor S
    else return __builtin_amdgcn_ds_bpermute((lane ^ S) << 2, v);
}

// Bitonic network over R * 64 keys held R per lane (element r * 64 + lane in
// v[r]): merge steps of block size SIZE from stride STRIDE down to 1. A block
// sorts ascending when (element & SIZE) == 0; in each pair the lower element
// keeps the minimum of an ascending block. Strides below 64 pair lanes
// (lane_xor), larger ones pair registers of one lane.
template <int R, int SIZE, int STRIDE>
__device__ __forceinline__ void bitonic_merge(int (&v)[R], int lane) {
    if constexpr (STRIDE >= kWave) {
        constexpr int RS = STRIDE / kWave;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if ((r & RS) == 0) {
                const bool asc = ((r * kWave) & SIZE) == 0;
                const int lo = min(v[r], v[r | RS]), hi = max(v[r], v[r | RS]);
                v[r] = asc ? lo : hi;
                v[r | RS] = asc ? hi : lo;
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int p = lane_xor<STRIDE>(v[r], lane);
            const bool asc = ((r * kWave + lane) & SIZE) == 0;
            const bool lower = (lane & STRIDE) == 0;
            v[r] = (asc == lower) ? min(v[r], p) : max(v[r], p);
        }
    }
    if constexpr (STRIDE > 1) bitonic_merge<R, SIZE, STRIDE / 2>(v, lane);
}
template <int R, int SIZE>
__device__ __forceinline__ void bitonic_sort(int (&v)[R], int lane) {
    if constexpr (SIZE > 2) bitonic_sort<R, SIZE / 2>(v, lane);
    bitonic_merge<R, SIZE, SIZE / 2>(v, lane);
}

// Sorts the n <= R * 64 distinct keys keys[0..n) in registers (padded with
// INT_MAX, which no particle index reaches) and stores them ascending to
// out[0..n) (out may alias keys).
template <int R>
__device__ __forceinline__ void sort_store(const int32_t* keys, int n, int32_t* out, int lane) {
    int v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = r * kWave + lane < n ? keys[r * kWave + lane] : INT_MAX;
    bitonic_sort<R, R * kWave>(v, lane);
#pragma unroll
    for (int r = 0; r < R; ++r)
        if (r * kWave + lane < n) out[r * kWave + lane] = v[r];
}

// Rows longer than this leave the row kernels unsorted; k_sort_long_rows
// sorts them afterwards, so the row kernels keep the registers of two keys
// per lane.
constexpr int kShortRow = 2 * kWave;

// Writes the n distinct keys of a wave's LDS list to out[0..n): sorted
// ascending when n <= kShortRow, as they are otherwise.
__device__ __forceinline__ void store_ranked(const int32_t* keys, int n, int32_t* __restrict__ out, int lane) {
    if (n <= kWave) {
        sort_store<1>(keys, n, out, lane);
    } else if (n <= kShortRow) {
        sort_store<2>(keys, n, out, lane);
    } else {
        for (int e = lane; e < n; e += kWave) out[e] = keys[e];
    }
}

// Sorts, in place, every row of the CSR longer than kShortRow (at most
// DCPSE_MAX_ROW = 1024 entries). Each wavefront reads 64 row lengths at a
// time and sorts the long ones among them in registers, up to 16 keys per lane.
__global__ __launch_bounds__(kRowWaves * kWave) void k_sort_long_rows(int64_t n_rows,
                                                                      const int64_t* __restrict__ row_ptr,
                                                                      int32_t* col) {
    static_assert(DCPSE_MAX_ROW <= 16 * kWave, "the row sort covers at most 1024 keys");
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * kRowWaves + (threadIdx.x >> 6);
    const int64_t nw = (int64_t)gridDim.x * kRowWaves;
    for (int64_t base = wave * kWave; base < n_rows; base += nw * kWave) {
        const int64_t p = base + lane;
        const int64_t rs_l = p < n_rows ? row_ptr[p] : 0;
        const int len_l = p < n_rows ? (int)(row_ptr[p + 1] - rs_l) : 0;
        unsigned long long m = __ballot(len_l > kShortRow);
        while (m) {
            const int j = __builtin_ctzll(m);
            m &= m - 1;
            const int64_t rs = readlane_i64(rs_l, j);
            const int n = min(__builtin_amdgcn_readlane(len_l, j), DCPSE_MAX_ROW);
            int32_t* row = col + rs;
            if (n <= 4 * kWave) sort_store<4>(row, n, row, lane);
            else if (n <= 8 * kWave) sort_store<8>(row, n, row, lane);
            else sort_store<16>(row, n, row, lane);
        }
    }
}

// The distance test of a candidate at xq against xp (the minimum image in
// periodic dimensions): the one formula of every support kernel.
template <int DIM>
__device__ __forceinline__ bool within_cut(const double* xp, const double* xq, const CellGrid& g, double r2) {
    double d[3];
#pragma unroll
    for (int dd = 0; dd < DIM; ++dd)
        d[dd] = min_image_r(xp[dd] - xq[dd], g.len[dd], g.ilen[dd], (g.periodic >> dd) & 1u);
    double d2 = d[DIM - 1] * d[DIM - 1];
#pragma unroll
    for (int dd = DIM - 2; dd >= 0; --dd) d2 = fma(d[dd], d[dd], d2);
    return d2 < r2;
}

// One wavefront per domain particle, or with list != NULL per particle
// list[1 ..] (list[0] = their number). FILL = false: count the support of p into
// counts[p] (and raise *overflow if it exceeds DCPSE_MAX_ROW). FILL = true:
// write the support of p, sorted ascending, to col[row_ptr[p] ..].
// The cells within k_d = ceil(rcut_p / cell edge) of p's cell in each
// dimension are scanned as rows along dimension 0: cells of one row are
// consecutive in the cell order, so a row is one contiguous candidate segment
// (two where a periodic wrap splits it). Up to 32 rows at a time, one segment
// per lane, are flattened into one candidate list by a prefix sum over the
// lanes.
template <int DIM, bool FILL>
__global__ __launch_bounds__(kRowWaves * kWave) void k_support_rows(
    const double* __restrict__ pos_dom, int64_t n_dom, int same_set, const int32_t* __restrict__ dom_self, const double* __restrict__ rcut, int rcut_pp,
    CellGrid g, const int64_t* __restrict__ cell_start, const CellRec* __restrict__ rec,
    int32_t* __restrict__ counts, int32_t* __restrict__ overflow, const int64_t* __restrict__ row_ptr,
    int32_t* __restrict__ col, const int32_t* __restrict__ list) {
    __shared__ int32_t buf[FILL ? kRowWaves : 1][FILL ? DCPSE_MAX_ROW : 1];
    __shared__ int32_t mark[kRowWaves][kWave];      // segment starting at a candidate of the round
    __shared__ long long seg_cst[kRowWaves][kWave];  // first cell slot of each segment
    __shared__ int32_t seg_ex[kRowWaves][kWave];     // candidates before each segment
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    const int64_t n_rows = list ? list[0] : n_dom;
    for (int64_t pi = (int64_t)blockIdx.x * kRowWaves + wv; pi < n_rows; pi += (int64_t)gridDim.x * kRowWaves) {
        const int64_t p = list ? list[1 + pi] : pi;
        double xp[3];
        int c[3] = {0, 0, 0};
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            xp[d] = pos_dom[d * n_dom + p];
            c[d] = cell_of(xp[d], d, g);
        }
        const double r = rcut_pp ? rcut[p] : rcut[0];
        // the reference particle skipped in this row (VL_SKIP_REF_PART): p
        // itself for one set, its support index for a subset domain
        const int self_q = same_set ? (int)p : (dom_self ? dom_self[p] : -1);
        const double r2 = r * r;
        int kd[3] = {0, 0, 0};
#pragma unroll
        for (int d = 0; d < DIM; ++d) kd[d] = min((int)ceil(r / g.cs[d]), g.kmax[d]);
        const int ny = 2 * kd[1] + 1;
        const int rows = DIM == 3 ? ny * (2 * kd[2] + 1) : ny;
        int nacc = 0;
        for (int rb = 0; rb < rows; rb += kWave / 2) {
            // lane 2i (+1): row rb + i (its part past a periodic wrap)
            long long cst = 0;
            int ccnt = 0;
            const int row = rb + (lane >> 1), part = lane & 1;
            if (row < rows) {
                const int o1 = row % ny - kd[1];
                const int o2 = DIM == 3 ? row / ny - kd[2] : 0;
                int cy = c[1] + o1, cz = DIM == 3 ? c[2] + o2 : 0;
                bool ok = true;
                if ((g.periodic >> 1) & 1u) cy = (cy % g.nc[1] + g.nc[1]) % g.nc[1];
                else ok &= cy >= 0 && cy < g.nc[1];
                if (DIM == 3) {
                    if ((g.periodic >> 2) & 1u) cz = (cz % g.nc[2] + g.nc[2]) % g.nc[2];
                    else ok &= cz >= 0 && cz < g.nc[2];
                }
                int xa = c[0] - kd[0], xb = c[0] + kd[0];
                if (g.periodic & 1u) {
                    if (xa < 0) {
                        if (part == 0) xa += g.nc[0], xb = g.nc[0] - 1;
                        else xa = 0;
                    } else if (xb >= g.nc[0]) {
                        if (part == 0) xb = g.nc[0] - 1;
                        else xa = 0, xb -= g.nc[0];
                    } else if (part == 1) {
                        ok = false;
                    }
                } else {
                    xa = max(xa, 0);
                    xb = min(xb, g.nc[0] - 1);
                    ok &= part == 0;
                }
                if (ok && xa <= xb) {
                    const int64_t lin = (int64_t)g.nc[0] * ((int64_t)cy + (int64_t)g.nc[1] * cz);
                    cst = cell_start[lin + xa];
                    ccnt = (int)(cell_start[lin + xb + 1] - cst);
                }
            }
            // inclusive prefix over lanes of the candidate counts
            const int incl = wave_incl_scan(ccnt);
            const int total = __builtin_amdgcn_readlane(incl, 63);
            const int excl = incl - ccnt;
            seg_cst[wv][lane] = cst;
            seg_ex[wv][lane] = excl;
            // segment of candidate k: the last non-empty segment starting at
            // or before k. Each round marks the segments that start inside its
            // 64 candidates, a prefix maximum spreads them, and a candidate
            // before the round's first start continues the previous segment.
            int carry = 0;
            for (int base = 0; base < total; base += kWave) {
                const int k = min(base + lane, total - 1);
                mark[wv][lane] = -1;
                wave_lds_sync();
                if (ccnt > 0 && excl >= base && excl < base + kWave) mark[wv][excl - base] = lane;
                wave_lds_sync();
                const int seg = max(wave_incl_max(mark[wv][lane]), carry);
                carry = __builtin_amdgcn_readlane(seg, 63);
                const long long s_cst = seg_cst[wv][seg];
                const int s_ex = seg_ex[wv][seg];
                const int64_t slot = s_cst + (k - s_ex);
                const CellRec cand = rec[slot];
                const int q = cand.id;
                const bool take = (base + lane < total) && q != self_q && within_cut<DIM>(xp, cand.x, g, r2);
                const unsigned long long m = __ballot(take);
                if (FILL) {
                    const int at = nacc + lane_prefix(m);
                    if (take && at < DCPSE_MAX_ROW) buf[wv][at] = q;
                }
                nacc += __popcll(m);
            }
        }
        if (!FILL) {
            if (lane == 0) {
                counts[p] = nacc;
                if (nacc > DCPSE_MAX_ROW) atomicOr(overflow, 1);
            }
        } else {
            wave_lds_sync();
            const int64_t rs = row_ptr[p];
            const int n = min(nacc, DCPSE_MAX_ROW);
            if ((int64_t)nacc != row_ptr[p + 1] - rs) {
                if (lane == 0) atomicOr(overflow, 2);
            } else {
                store_ranked(buf[wv], n, col + rs, lane);
            }
            wave_lds_sync();
        }
    }
}

// ---- one set: a wavefront per group of neighbouring particles --------------
// A group is the particles of one home cell. With one cut-off the home cells
// are the cells of the list (edge >= rcut) and a group's candidates those of
// the 3^dim cells around it; with a cut-off per particle the home cells come
// in levels by cut-off (HomeLevels) and the candidates from the cells within
// the group's largest cut-off of its bounding box. Cells along dimension 0 are
// consecutive in the cell order, so a row of cells is one contiguous segment of
// candidates (two across a periodic wrap).
// The count pass (k_group_pairs) keeps the candidates within reach of the
// group's bounding box, sorts their indices once, and tests every particle of
// the group against them: it stores the group's sorted candidate list and, per
// particle, which of them it takes (one bit each). The fill (k_group_rows)
// writes a particle's row as the marked entries of its group's list, which are
// in ascending order as they stand: no distance work and no sort per row.
// Particles of groups with more candidates than the list holds are left to
// k_support_rows. All decide by within_cut (k_group_pairs wherever FP32 leaves
// the outcome open), so the results are the same.

// Cell c's coordinates (cells number below 2^31, see make_grid).
template <int DIM>
__device__ __forceinline__ void cell_coords(const CellGrid& g, int64_t c, int (&cc)[3]) {
    unsigned rem = (unsigned)c;
    cc[0] = cc[1] = cc[2] = 0;
#pragma unroll
    for (int d = 0; d < DIM - 1; ++d) {
        const unsigned q = rem / (unsigned)g.nc[d];
        cc[d] = (int)(rem - q * (unsigned)g.nc[d]);
        rem = q;
    }
    cc[DIM - 1] = (int)rem;
}

// The candidate segments of cell c: lane 2i (+1) gets row i of the 3^(dim-1)
// rows of three cells along dimension 0 (its part past a periodic wrap), as
// the first cell slot cst and the length ccnt (0 for no segment).
template <int DIM>
__device__ __forceinline__ void cell_segments(const CellGrid& g, const int64_t* __restrict__ cell_start,
                                              const int (&cc)[3], int lane, int64_t& cst, int& ccnt) {
    constexpr int ROWS = DIM == 3 ? 9 : 3;
    cst = 0;
    ccnt = 0;
    const int row = lane >> 1, part = lane & 1;
    if (row >= ROWS) return;
    int cy = cc[1] + row % 3 - 1, cz = DIM == 3 ? cc[2] + row / 3 - 1 : 0;
    bool ok = true;
    if ((g.periodic >> 1) & 1u) cy += cy < 0 ? g.nc[1] : cy >= g.nc[1] ? -g.nc[1] : 0;
    else ok &= cy >= 0 && cy < g.nc[1];
    if (DIM == 3) {
        if ((g.periodic >> 2) & 1u) cz += cz < 0 ? g.nc[2] : cz >= g.nc[2] ? -g.nc[2] : 0;
        else ok &= cz >= 0 && cz < g.nc[2];
    }
    int xa = cc[0] - 1, xb = cc[0] + 1;
    if (g.periodic & 1u) {
        if (xa < 0) {
            if (part == 0) xa += g.nc[0], xb = g.nc[0] - 1;
            else xa = 0;
        } else if (xb >= g.nc[0]) {
            if (part == 0) xb = g.nc[0] - 1;
            else xa = 0, xb -= g.nc[0];
        } else if (part == 1) {
            ok = false;
        }
    } else {
        xa = max(xa, 0);
        xb = min(xb, g.nc[0] - 1);
        ok &= part == 0;
    }
    if (ok && xa <= xb) {
        const int64_t lin = (int64_t)g.nc[0] * ((int64_t)cy + (int64_t)g.nc[1] * cz);
        cst = cell_start[lin + xa];
        ccnt = (int)(cell_start[lin + xb + 1] - cst);
    }
}

// Candidates are handled in coordinates relative to the group's centre, in
// units of its largest cut-off, in FP32: there |a - b|^2 is within 4e-6 of the
// FP64 value for particles up to kMaxReach from the centre whose positions lie
// within kMaxOffset cut-offs of the origin (FP64 then resolves 1e-9 cut-offs),
// so outside kPairTol around a particle's squared cut-off it decides the pair
// and inside the FP64 formula does.
constexpr float kPairTol = 2e-5f;
constexpr float kMaxReach = 8.0f;
constexpr double kMaxOffset = 1e7;
constexpr int kPairWaves = 4;  // groups (wavefronts) per block

// v of lane ^ X for the lane exchanges of the sorting network.
template <int X>
__device__ __forceinline__ int lane_xor_key(int v, int lane) {
    if constexpr (X == 1 || X == 2 || X == 8) return lane_xor<X>(v, lane);
    else if constexpr (X == 3) return __builtin_amdgcn_update_dpp(0, v, 0x1B, 0xF, 0xF, false);    // quad_perm 3,2,1,0
    else if constexpr (X == 7) return __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, false);   // row_half_mirror
    else if constexpr (X == 15) return __builtin_amdgcn_update_dpp(0, v, 0x140, 0xF, 0xF, false);  // row_mirror
    else if constexpr (X == 4) return lane_xor_key<3>(lane_xor_key<7>(v, lane), lane);
    else if constexpr (X == 31) return __builtin_amdgcn_ds_swizzle(v, 0x1F | (31 << 10));
    else return __builtin_amdgcn_ds_bpermute((lane ^ X) << 2, v);
}

// The smaller of v and p in lanes with sel = INT_MIN, the larger with INT_MAX
// (the median of three: one instruction).
__device__ __forceinline__ int pick(int v, int p, int sel) { return max(min(v, p), min(max(v, p), sel)); }

constexpr int log2_c(int x) { return x <= 1 ? 0 : 1 + log2_c(x / 2); }

// Half-cleaner of stride S over elements e = lane * R + r (lower index keeps
// the smaller), then the smaller strides.
template <int R, int S>
__device__ __forceinline__ void clean_keys(int (&v)[R], const int (&sel)[6], int lane) {
    if constexpr (S >= R) {
        constexpr int X = S / R;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (X == 16) {  // both rows of a pair side by side in one exchange
                const auto x = __builtin_amdgcn_permlane16_swap((unsigned)v[r], (unsigned)v[r], false, false);
                v[r] = pick((int)x[0], (int)x[1], sel[4]);
            } else {
                v[r] = pick(v[r], lane_xor_key<X>(v[r], lane), sel[log2_c(X)]);
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; ++r)
            if ((r & S) == 0) {
                const int a = v[r], b = v[r | S];
                v[r] = min(a, b);
                v[r | S] = max(a, b);
            }
    }
    if constexpr (S > 1) clean_keys<R, S / 2>(v, sel, lane);
}

// Ascending sort of R * 64 keys held as element lane * R + r: merges of
// doubling blocks, each opened by a mirrored exchange (element i of the block
// with SIZE - 1 - i) so that every comparison points the same way. With a
// lane's R keys adjacent, the short strides, which are the most frequent,
// stay in registers.
template <int R, int SIZE>
__device__ __forceinline__ void sort_keys(int (&v)[R], const int (&sel)[6], int lane) {
    if constexpr (SIZE > 2) sort_keys<R, SIZE / 2>(v, sel, lane);
    if constexpr (SIZE <= R) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int m = r ^ (SIZE - 1);
            if (r < m) {
                const int a = v[r], b = v[m];
                v[r] = min(a, b);
                v[m] = max(a, b);
            }
        }
    } else {
        constexpr int X = SIZE / R - 1;
        int p[R];
#pragma unroll
        for (int r = 0; r < R; ++r) p[r] = lane_xor_key<X>(v[R - 1 - r], lane);
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = pick(v[r], p[r], sel[log2_c((X + 1) / 2)]);
    }
    if constexpr (SIZE >= 4) clean_keys<R, SIZE / 4>(v, sel, lane);
}

// Minimum over the 64 lanes, in every lane.
__device__ __forceinline__ float wave_min_f(float v) {
    auto d = [](float x, auto ctrl) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xF, 0xF, true));
    };
    v = fminf(v, d(v, std::integral_constant<int, 0xB1>()));
    v = fminf(v, d(v, std::integral_constant<int, 0x4E>()));
    v = fminf(v, d(v, std::integral_constant<int, 0x141>()));
    v = fminf(v, d(v, std::integral_constant<int, 0x140>()));
    auto l = [&](int lane) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane)); };
    return fminf(fminf(l(0), l(16)), fminf(l(32), l(48)));
}

__device__ __forceinline__ float readlane_f(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// old with lane l's value replaced by the wave-uniform v (v_writelane).
extern "C" __device__ int dcpse_writelane(int v, int l, int old) __asm("llvm.amdgcn.writelane.i32");

// The groups of a pass and where its results go.
struct Groups {
    int64_t n;                   // particles
    const double* pos;           // by particle
    const double* rcut;          // one, or one per particle (PP)
    CellGrid g;                  // candidate cells
    const int64_t* cell_start;
    const CellRec* rec;          // by candidate cell
    const int64_t* home_start;   // by home cell
    const CellRec* home;
    const int32_t* group_cell;   // home cell of each group, or NULL: every home cell is a group
    const int64_t* n_groups;     // on the device, or NULL: max_groups
    int64_t max_groups;          // groups with a list; the others' particles are spilled
    int32_t* counts;
    int32_t* flags;
    int32_t* ncand;              // candidates of a group, -1: spilled
    int32_t* lists;              // nws * 64 entries per group
    uint64_t* masks;             // nws words per home slot
    int nws;
    int32_t* spill;
};

// The group of this wavefront, -1 for none: consecutive groups, which share
// most candidates, on one XCD (blocks are dealt round-robin over the 8 XCDs).
__device__ __forceinline__ int64_t wave_group(const Groups& a) {
    const int64_t ng = a.n_groups ? *a.n_groups : a.max_groups;
    const int64_t per = (ng + 8 * kPairWaves - 1) / (8 * kPairWaves);  // blocks per XCD
    const int64_t i = blockIdx.x >> 3;
    if (i >= per) return -1;
    const int64_t gi =
        ((blockIdx.x & 7) * per + i) * kPairWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    return gi < ng ? gi : -1;
}

// What a wave knows of its group: centre, unit of length, particles.
struct PairGroup {
    double ctr[3];
    double unit, iunit;
    int64_t pst;
    int np, total;  // particles; candidates kept
};

// Position x (component d) relative to the group's centre: the image nearest
// to it in a periodic dimension. The period exceeds the home cell and two
// cut-offs, so wherever a pair is within the cut-off these images are the ones
// its minimum image takes.
__device__ __forceinline__ float relative(const PairGroup& pg, const CellGrid& g, double x, int d) {
    // an open dimension has period 0: no select per lane
    const bool wraps = (g.periodic >> d) & 1u;
    return (float)(min_image_r(x - pg.ctr[d], wraps ? g.len[d] : 0.0, wraps ? g.ilen[d] : 0.0, true) * pg.iunit);
}

// Sorts the group's pg.total <= R * 64 candidate indices (in the wave's LDS
// list), stores them and tests the group's particles against them.
template <int DIM, int R, bool PP>
__device__ __forceinline__ void pair_tests(const Groups& a, const PairGroup& pg, int64_t gi, int32_t* keys, int lane) {
    const int64_t n = a.n;
    int32_t* __restrict__ list = a.lists + gi * a.nws * kWave;
    int key[R];
    int sel[6];
#pragma unroll
    for (int b = 0; b < 6; ++b) sel[b] = (lane >> b) & 1 ? INT_MAX : INT_MIN;
#pragma unroll
    for (int r = 0; r < R; ++r) key[r] = lane * R + r < pg.total ? keys[lane * R + r] : INT_MAX;
    sort_keys<R, R * kWave>(key, sel, lane);
    // to element r * 64 + lane, so that a mask word covers 64 consecutive entries
    wave_lds_sync();
#pragma unroll
    for (int r = 0; r < R; ++r) keys[lane * R + r] = key[r];
    wave_lds_sync();
    float cx[R][DIM];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        key[r] = keys[r * kWave + lane];
        const bool have = r * kWave + lane < pg.total;
        const int64_t q = have ? key[r] : 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const float x = relative(pg, a.g, a.pos[d * n + q], d);
            cx[r][d] = have ? x : 1e18f;  // padding is out of reach
        }
        if (have) list[r * kWave + lane] = key[r];
    }
    const int nw = (pg.total + kWave - 1) >> 6;
    for (int i0 = 0; i0 < pg.np; i0 += kWave) {
        const int m64 = min(kWave, pg.np - i0);
        int pid = 0;
        float xp[DIM];
        float t2 = 1.0f;  // squared cut-off
        {
            const CellRec h = a.home[pg.pst + i0 + min(lane, m64 - 1)];
            pid = h.id;
#pragma unroll
            for (int d = 0; d < DIM; ++d) xp[d] = relative(pg, a.g, h.x[d], d);
            if (PP) {
                const double rc = a.rcut[pid];
                const float t = (float)(rc * pg.iunit);
                t2 = rc > 0.0 ? t * t : -1.0f;
            }
        }
        int cnt = 0;
        constexpr int PER = kWave / R;  // particles whose mask words fill the lanes
        for (int ib = 0; ib < m64; ib += PER) {
            const int ie = min(PER, m64 - ib);
            int wlo = 0, whi = 0;
            for (int k = 0; k < ie; ++k) {
                const int i = ib + k;
                const int p = __builtin_amdgcn_readlane(pid, i);
                float x[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) x[d] = readlane_f(xp[d], i);
                const float t = PP ? readlane_f(t2, i) : 1.0f;
                const float tin = t - kPairTol, tout = t + kPairTol;
                int nacc = 0;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if (r > R / 2 && r >= nw) break;  // the last words are often empty
                    float d2 = 0.0f;
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        const float u = cx[r][d] - x[d];
                        d2 = fmaf(u, u, d2);
                    }
                    unsigned long long m = __ballot(d2 < tout) & ~__ballot(key[r] == p);
                    const unsigned long long open = m & __ballot(d2 > tin);
                    if (open) {  // rare: the FP64 formula on the positions themselves
                        double xa[3], xb[3];
                        const bool mine = (open >> lane) & 1u;
                        const int64_t q = mine ? key[r] : p;
                        const double rc = a.rcut[PP ? p : 0];
#pragma unroll
                        for (int d = 0; d < DIM; ++d) {
                            xa[d] = a.pos[d * n + p];
                            xb[d] = a.pos[d * n + q];
                        }
                        m = (m & ~open) | (open & __ballot(within_cut<DIM>(xa, xb, a.g, rc * rc)));
                    }
                    nacc += __popcll(m);
                    wlo = dcpse_writelane((int)m, k * R + r, wlo);
                    whi = dcpse_writelane((int)(m >> 32), k * R + r, whi);
                }
                cnt = dcpse_writelane(nacc, i, cnt);
            }
            if (lane < ie * R && lane % R < nw)
                a.masks[(pg.pst + i0 + ib + lane / R) * a.nws + lane % R] =
                    ((uint64_t)(unsigned)whi << 32) | (unsigned)wlo;
        }
        if (lane < m64) {
            a.counts[pid] = cnt;
            if (cnt > DCPSE_MAX_ROW) atomicOr(a.flags, 1);
        }
    }
}

// Count pass: one wavefront per group (see above). Groups beyond max_groups,
// with more than nws * 64 candidates or with a particle that FP32 would
// resolve too coarsely go to the spill list (spill[0] particles at spill[1 ..]).
// RMAX * 64 >= nws * 64 bounds the registers.
//
// Bound by VALU issue: 342 candidates per cell of the 128^3 set with 10%
// removed (rcut 2.4 spacings) shrink to about 170 within reach of the
// particles' bounding box, are sorted in 200-odd instructions, and a pair
// test costs 9 instructions per 64 pairs with the candidates in registers and
// the particle in scalar registers. 0.51 ms there (1.89M particles); FP64
// tests of every candidate from LDS took 1.14 ms, and with them the fill,
// which then sorted every row, 0.96 ms instead of 0.22 ms (k_group_rows).
// With a cut-off per particle (PP; 490,000 particles, spacing 4 : 1): 0.27 ms
// and a fill of 0.11 ms, against 1.08 and 1.22 ms of k_support_rows, whose
// wavefronts each flatten and test the candidates of one particle.
template <int DIM, int RMAX, bool PP>
__global__ __launch_bounds__(kPairWaves * kWave) void k_group_pairs(const Groups a, const HomeLevels h) {
    __shared__ __align__(16) int32_t kbuf[kPairWaves][RMAX * kWave];
    __shared__ int32_t marks[PP ? kPairWaves : 1][PP ? 4 * kWave : 1];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t gi = wave_group(a);
    if (gi < 0) return;  // whole wavefront
    const int64_t c = a.group_cell ? a.group_cell[gi] : gi;
    const CellGrid& g = a.g;
    PairGroup pg;
    pg.pst = a.home_start[c];
    pg.np = (int)(a.home_start[c + 1] - pg.pst);
    if (pg.np == 0) return;  // never looked at by the fill either
    int cc[3];
    if constexpr (PP) {
        int l = 0;
#pragma unroll
        for (int i = 1; i < kMaxLevels; ++i)
            if (i < h.n && c >= h.first[i]) l = i;
        const CellGrid& hg = h.g[l];
        cell_coords<DIM>(hg, c - h.first[l], cc);
#pragma unroll
        for (int d = 0; d < DIM; ++d) pg.ctr[d] = hg.lo[d] + (cc[d] + 0.5) * hg.cs[d];
        float rm = 0.0f;
        for (int i0 = 0; i0 < pg.np; i0 += kWave)
            if (i0 + lane < pg.np) rm = fmaxf(rm, (float)a.rcut[a.home[pg.pst + i0 + lane].id]);
        // a little above the largest cut-off: every particle's lies within the unit
        pg.unit = fmax((double)(-wave_min_f(-rm)) * 1.0000005, 1e-6 * h.rtop);
    } else {
        cell_coords<DIM>(g, c, cc);
#pragma unroll
        for (int d = 0; d < DIM; ++d) pg.ctr[d] = g.lo[d] + (cc[d] + 0.5) * g.cs[d];
        pg.unit = a.rcut[0];
    }
    pg.iunit = 1.0 / pg.unit;
    const double xmax = kMaxOffset * pg.unit;
    // bounding box of the group
    float lo[DIM], hi[DIM];
    bool wild = gi >= a.max_groups;
#pragma unroll
    for (int d = 0; d < DIM; ++d) lo[d] = hi[d] = 1e30f;  // hi: of the negated coordinate
    for (int i0 = 0; i0 < pg.np; i0 += kWave) {
        const CellRec r = a.home[pg.pst + min(i0 + lane, pg.np - 1)];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            wild |= fabs(r.x[d]) > xmax;
            const float x = relative(pg, g, r.x[d], d);
            lo[d] = fminf(lo[d], x);
            hi[d] = fminf(hi[d], -x);
        }
    }
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        lo[d] = wave_min_f(lo[d]);
        hi[d] = -wave_min_f(hi[d]);
        wild |= !(lo[d] >= -kMaxReach && hi[d] <= kMaxReach);
    }
    int nacc = 0;
    // keeps those of four candidates per lane that are within reach of the box
    // (left of them: the last ones past the end of a list are skipped)
    auto take4 = [&](const int64_t (&slot)[4], const bool (&have)[4], int left) {
        CellRec r[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (j * kWave < left) r[j] = a.rec[slot[j]];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (j * kWave >= left) break;
            float d2 = 0.0f;  // squared distance to the box
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                wild |= fabs(r[j].x[d]) > xmax;
                const float x = relative(pg, g, r[j].x[d], d);
                const float t = fmaxf(fmaxf(lo[d] - x, x - hi[d]), 0.0f);
                d2 = fmaf(t, t, d2);
            }
            const bool keep = have[j] & (d2 < 1.0f + 4.0f * kPairTol);
            const unsigned long long m = __ballot(keep);
            const int at = nacc + lane_prefix(m);
            if (keep && at < RMAX * kWave) kbuf[wv][at] = r[j].id;
            nacc += __popcll(m);
        }
    };
    bool spilled = __ballot(wild) != 0;
    if (!spilled) {
        if constexpr (PP) {
            // cells within the cut-off of the box, a dimension at a time (unwrapped)
            int ia[3] = {0, 0, 0}, ib[3] = {0, 0, 0};
            bool whole[3] = {false, false, false};
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                const double ics = 1.0 / g.cs[d], at = pg.ctr[d] - g.lo[d];
                ia[d] = (int)floor((at + ((double)lo[d] - 1.0001) * pg.unit) * ics);
                ib[d] = (int)floor((at + ((double)hi[d] + 1.0001) * pg.unit) * ics);
                if (!((g.periodic >> d) & 1u)) {
                    ia[d] = min(max(ia[d], 0), g.nc[d] - 1);
                    ib[d] = min(max(ib[d], 0), g.nc[d] - 1);
                } else if (ib[d] - ia[d] + 1 >= g.nc[d]) {
                    whole[d] = true;
                    ia[d] = 0;
                    ib[d] = g.nc[d] - 1;
                }
            }
            const int ny = ib[1] - ia[1] + 1;
            const int rows = DIM == 3 ? ny * (ib[2] - ia[2] + 1) : ny;
            // distance of the box from the slab of cell index v of dimension d
            auto gap = [&](int v, int d) {
                const double s0 = (g.lo[d] + v * g.cs[d] - pg.ctr[d]) * pg.iunit;
                const float below = (float)(s0 - hi[d]), above = (float)(lo[d] - (s0 + g.cs[d] * pg.iunit));
                float t = fmaxf(below, above) - 1e-4f;
                if (!((g.periodic >> d) & 1u)) {  // the outermost cells hold what lies outside
                    if (v == 0) t = above - 1e-4f;
                    if (v == g.nc[d] - 1) t = v == 0 ? 0.0f : below - 1e-4f;
                }
                return whole[d] ? 0.0f : fmaxf(t, 0.0f);
            };
            for (int rb = 0; rb < rows; rb += kWave / 2) {
                // lane 2i (+1): row rb + i (its part past a periodic wrap)
                int64_t cst = 0;
                int ccnt = 0;
                const int row = rb + (lane >> 1), part = lane & 1;
                if (row < rows) {
                    const int oz = DIM == 3 ? (int)((unsigned)row / (unsigned)ny) : 0;
                    int cy = ia[1] + row - oz * ny, cz = ia[2] + oz;
                    const float gy = gap(cy, 1), gz = DIM == 3 ? gap(cz, 2) : 0.0f;
                    const float rest = 1.0001f - fmaf(gy, gy, gz * gz);
                    if (rest > 0.0f) {
                        const double half = (double)sqrtf(rest) + 1e-4;
                        const double at = pg.ctr[0] - g.lo[0], ics = 1.0 / g.cs[0];
                        int xa = ia[0], xb = ib[0];
                        if (!whole[0]) {  // (ia, ib are clamped in an open dimension: so are these)
                            xa = min(max(xa, (int)floor((at + (lo[0] - half) * pg.unit) * ics)), ib[0]);
                            xb = max(min(xb, (int)floor((at + (hi[0] + half) * pg.unit) * ics)), ia[0]);
                        }
                        if ((g.periodic >> 1) & 1u) cy += cy < 0 ? g.nc[1] : cy >= g.nc[1] ? -g.nc[1] : 0;
                        if (DIM == 3 && ((g.periodic >> 2) & 1u))
                            cz += cz < 0 ? g.nc[2] : cz >= g.nc[2] ? -g.nc[2] : 0;
                        bool ok = xa <= xb;
                        if (xa < 0) {  // wraps below: [xa + nc, nc) and [0, xb]
                            if (xb < 0) xa += g.nc[0], xb += g.nc[0], ok &= part == 0;
                            else if (part == 0) xa += g.nc[0], xb = g.nc[0] - 1;
                            else xa = 0;
                        } else if (xb >= g.nc[0]) {
                            if (xa >= g.nc[0]) xa -= g.nc[0], xb -= g.nc[0], ok &= part == 0;
                            else if (part == 0) xb = g.nc[0] - 1;
                            else xa = 0, xb -= g.nc[0];
                        } else {
                            ok &= part == 0;
                        }
                        if (ok) {
                            const int64_t lin = (int64_t)g.nc[0] * ((int64_t)cy + (int64_t)g.nc[1] * cz);
                            cst = a.cell_start[lin + xa];
                            ccnt = (int)(a.cell_start[lin + xb + 1] - cst);
                        }
                    }
                }
                const int incl = wave_incl_scan(ccnt);
                const int total = __builtin_amdgcn_readlane(incl, 63);
                const int excl = incl - ccnt;
                const int delta = (int)cst - excl;  // slot of candidate k of this segment: k + delta
                // segment of candidate k: the last non-empty one starting at or
                // before it. Each round marks the starts inside its 256
                // candidates, a prefix maximum spreads them, and the last one
                // carries over.
                int32_t* mark = marks[wv];
                int carry = 0;
                for (int base = 0; base < total; base += 4 * kWave) {
                    wave_lds_sync();
#pragma unroll
                    for (int j = 0; j < 4; ++j) mark[j * kWave + lane] = -1;
                    wave_lds_sync();
                    if (ccnt > 0 && excl >= base && excl < base + 4 * kWave) mark[excl - base] = lane;
                    wave_lds_sync();
                    int64_t slot[4];
                    bool have[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int seg = max(wave_incl_max(mark[j * kWave + lane]), carry);
                        carry = __builtin_amdgcn_readlane(seg, 63);
                        const int k = base + j * kWave + lane;
                        have[j] = k < total;
                        const int dl = __builtin_amdgcn_ds_bpermute(seg << 2, delta);
                        slot[j] = have[j] ? k + dl : 0;
                    }
                    take4(slot, have, total - base);
                }
            }
        } else {
            int64_t cst;
            int ccnt;
            cell_segments<DIM>(g, a.cell_start, cc, lane, cst, ccnt);
            const int incl = wave_incl_scan(ccnt);
            const int total = __builtin_amdgcn_readlane(incl, 63);
            const int excl = incl - ccnt;
            const int delta = (int)cst - excl;  // slot of candidate k of this segment: k + delta
            const unsigned long long segs = __ballot(ccnt > 0);
            for (int base = 0; base < total; base += 4 * kWave) {
                int off[4] = {0, 0, 0, 0};
                for (unsigned long long m = segs; m; m &= m - 1) {
                    const int s = __builtin_ctzll(m);
                    const int ex = __builtin_amdgcn_readlane(excl, s);
                    const int dl = __builtin_amdgcn_readlane(delta, s);
#pragma unroll
                    for (int j = 0; j < 4; ++j) off[j] = base + j * kWave + lane >= ex ? dl : off[j];
                }
                int64_t slot[4];
                bool have[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int k = base + j * kWave + lane;
                    have[j] = k < total;
                    slot[j] = have[j] ? k + off[j] : 0;
                }
                take4(slot, have, total - base);
            }
        }
        spilled = nacc > a.nws * kWave || __ballot(wild) != 0;
    }
    if (spilled) {
        int at = 0;
        if (lane == 0) {
            at = 1 + atomicAdd(a.spill, pg.np);
            if (gi < a.max_groups) a.ncand[gi] = -1;
        }
        at = __builtin_amdgcn_readfirstlane(at);
        for (int i = lane; i < pg.np; i += kWave) a.spill[at + i] = a.home[pg.pst + i].id;
        return;
    }
    if (lane == 0) a.ncand[gi] = nacc;
    pg.total = nacc;
    wave_lds_sync();
    if (nacc <= RMAX / 4 * kWave) pair_tests<DIM, RMAX / 4, PP>(a, pg, gi, kbuf[wv], lane);
    else if (nacc <= RMAX / 2 * kWave) pair_tests<DIM, RMAX / 2, PP>(a, pg, gi, kbuf[wv], lane);
    else pair_tests<DIM, RMAX, PP>(a, pg, gi, kbuf[wv], lane);
}

// The rows of a group's particles from its candidate list and the take masks.
template <int R>
__device__ __forceinline__ void pair_rows(const Groups& a, int64_t gi, int64_t pst, int np, int total,
                                          const int64_t* __restrict__ row_ptr, int32_t* __restrict__ col, int lane) {
    const int32_t* __restrict__ list = a.lists + gi * a.nws * kWave;
    int key[R];
#pragma unroll
    for (int r = 0; r < R; ++r) key[r] = r * kWave + lane < total ? list[r * kWave + lane] : 0;
    const int nw = (total + kWave - 1) >> 6;
    constexpr int PER = kWave / R;
    for (int i0 = 0; i0 < np; i0 += kWave) {
        const int m64 = min(kWave, np - i0);
        int64_t rs = 0;
        int len = 0;
        if (lane < m64) {
            const int pid = a.home[pst + i0 + lane].id;
            rs = row_ptr[pid];
            len = (int)(row_ptr[pid + 1] - rs);
        }
        for (int ib = 0; ib < m64; ib += PER) {
            const int ie = min(PER, m64 - ib);
            uint64_t mw = 0;
            if (lane < ie * R && lane % R < nw) mw = a.masks[(pst + i0 + ib + lane / R) * a.nws + lane % R];
            for (int k = 0; k < ie; ++k) {
                const int64_t row = readlane_i64(rs, ib + k);
                const int n = __builtin_amdgcn_readlane(len, ib + k);
                uint64_t m[R];
                int tot = 0;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    m[r] = (uint64_t)readlane_i64((int64_t)mw, k * R + r);
                    tot += __popcll(m[r]);
                }
                if (tot != n) {  // counted on other positions
                    if (lane == 0) atomicOr(a.flags, 2);
                    continue;
                }
                int32_t* out = col + row;
                int at = 0;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if ((m[r] >> lane) & 1u) out[at + lane_prefix(m[r])] = key[r];
                    at += __popcll(m[r]);
                }
            }
        }
    }
}

// Fill pass over the groups that k_group_pairs listed: a wavefront per group,
// a masked store per 64 candidates of a row and nothing else; bound by the
// stores and the instructions that address them.
template <int RMAX>
__global__ __launch_bounds__(kPairWaves * kWave) void k_group_rows(const Groups a,
                                                                   const int64_t* __restrict__ row_ptr,
                                                                   int32_t* __restrict__ col) {
    const int lane = threadIdx.x & 63;
    const int64_t gi = wave_group(a);
    if (gi < 0 || gi >= a.max_groups) return;  // beyond: filled from positions
    const int64_t c = a.group_cell ? a.group_cell[gi] : gi;
    const int64_t pst = a.home_start[c];
    const int np = (int)(a.home_start[c + 1] - pst);
    if (np == 0) return;
    const int total = a.ncand[gi];
    if (total < 0) return;  // filled from positions
    if (total <= RMAX / 4 * kWave) pair_rows<RMAX / 4>(a, gi, pst, np, total, row_ptr, col, lane);
    else if (total <= RMAX / 2 * kWave) pair_rows<RMAX / 2>(a, gi, pst, np, total, row_ptr, col, lane);
    else pair_rows<RMAX>(a, gi, pst, np, total, row_ptr, col, lane);
}

// Cell edge about rmax / K: smaller cells than the cut-off shrink the scanned
// volume around a particle ((2k+1)^dim cells of edge rmax/K instead of 3^dim
// of edge rmax), and let particles with a smaller cut-off scan fewer cells.
// A periodic dimension needs at least 2k+1 cells; where the box is too small
// for that, the edge falls back to rmax (k = 1, at least 3 cells).
static dcpse_status make_grid(dcpse_ctx* ctx, int dim, const double* box_lo, const double* box_hi,
                              unsigned periodic, double rmax, int K, CellGrid* g) {
    if (!(rmax > 0.0) || !std::isfinite(rmax)) return fail(ctx, DCPSE_ERR_INVALID, "rcut must be > 0");
    g->ncell = 1;
    g->periodic = periodic;
    for (int d = 0; d < 3; ++d) {
        if (d < dim) {
            double len = box_hi[d] - box_lo[d];
            if (!(len > 0.0)) return fail(ctx, DCPSE_ERR_INVALID, "box_hi must exceed box_lo");
            int n = (int)std::floor(len * K / rmax);
            if (n < 1) n = 1;
            // keep the cell grid bounded (cells beyond ~2^26 add nothing but memory)
            while ((double)g->ncell * n > 6.7e7 && n / 2 >= 3) n /= 2;
            int kmax = (int)std::ceil(rmax / (len / n));
            if (((periodic >> d) & 1u) && n < 2 * kmax + 1) {
                n = (int)std::floor(len / rmax);
                if (n < 3)
                    return fail(ctx, DCPSE_ERR_INVALID,
                                "periodic dimension %d has %d cells of edge >= rcut (need 3)", d, n);
                kmax = 1;
            }
            g->nc[d] = n;
            g->kmax[d] = kmax;
            g->lo[d] = box_lo[d];
            g->len[d] = len;
            g->ilen[d] = 1.0 / len;
            g->cs[d] = len / n;
            g->ncell *= n;
        } else {
            g->nc[d] = 1; g->kmax[d] = 0; g->lo[d] = 0; g->len[d] = 1; g->ilen[d] = 1; g->cs[d] = 1;
        }
    }
    return DCPSE_OK;
}

// Per block: out[2b] = min and out[2b + 1] = max(0, max) of its share of
// v[0..n) (NaNs ignored).
constexpr int kMinMaxThreads = 256;
constexpr int kMinMaxBlocks = 256;
__global__ __launch_bounds__(kMinMaxThreads) void k_minmax(const double* __restrict__ v, int64_t n,
                                                          double* __restrict__ out) {
    __shared__ double smin[kMinMaxThreads], smax[kMinMaxThreads];
    const int t = threadIdx.x;
    double lo = v[0], hi = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * kMinMaxThreads + t; i < n; i += (int64_t)gridDim.x * kMinMaxThreads) {
        lo = fmin(lo, v[i]);
        hi = fmax(hi, v[i]);
    }
    smin[t] = lo;
    smax[t] = hi;
    __syncthreads();
    for (int off = kMinMaxThreads / 2; off > 0; off >>= 1) {
        if (t < off) {
            smin[t] = fmin(smin[t], smin[t + off]);
            smax[t] = fmax(smax[t], smax[t + off]);
        }
        __syncthreads();
    }
    if (t == 0) {
        out[2 * blockIdx.x] = smin[0];
        out[2 * blockIdx.x + 1] = smax[0];
    }
}

// Calls launch with the dimension and the register width of a mask of nws
// words as compile-time values.
template <typename F>
static void launch_groups(int dim, int nws, F launch) {
    auto width = [&](auto D) {
        if (nws <= 4) launch(D, std::integral_constant<int, 4>());
        else if (nws <= 8) launch(D, std::integral_constant<int, 8>());
        else if (nws <= 16) launch(D, std::integral_constant<int, 16>());
        else launch(D, std::integral_constant<int, 32>());
    };
    if (dim == 2) width(std::integral_constant<int, 2>());
    else width(std::integral_constant<int, 3>());
}

// Home cells of a set too sparse to fill them. A home cell takes 24 bytes and a
// few passes; up to this many groups are faster than a wavefront per particle
// (300,000 particles of 47 neighbours in one corner, us with groups / without:
// 4.8M cells 459 / 1268, 19M 863 / 1708, 38M 1385 / 2049) and the memory is no
// more than that of the cells make_grid allows (6.7e7 of 12 bytes); a box of 500
// cut-offs a side would have 2e8.
constexpr double kMaxHomeCells = 3.4e7;

// The home levels of a set with cut-offs in [rmin, rmax]: a level for every
// halving, as long as their cells number a few per particle.
static void make_levels(int dim, const double* box_lo, const double* box_hi, unsigned periodic, double rmin,
                        double rmax, int64_t n, HomeLevels* h) {
    h->n = 0;
    h->rtop = rmax;
    h->first[0] = 0;
    double total = 0.0, edge = kHomeEdge * rmax, top = rmax;
    for (int l = 0; l < kMaxLevels; ++l, edge *= 0.5, top *= 0.5) {
        if (l > 0 && !(rmin <= top)) break;  // no particle is this small
        CellGrid& g = h->g[l];
        g.periodic = periodic;
        double cells = 1.0;
        for (int d = 0; d < 3; ++d) {
            const double len = d < dim ? box_hi[d] - box_lo[d] : 1.0;
            const double k = d < dim ? std::min(std::max(std::ceil(len / edge), 1.0), 1e6) : 1.0;
            g.nc[d] = (int)k;
            g.kmax[d] = 0;
            g.lo[d] = d < dim ? box_lo[d] : 0.0;
            g.len[d] = len;
            g.ilen[d] = 1.0 / len;
            g.cs[d] = len / k;
            cells *= k;
        }
        if (total + cells > 4.0 * (double)n + 4096.0 && l > 0) break;
        total += cells;
        if (total > std::min(std::max(kMaxHomeCells, 4.0 * (double)n + 4096.0), 1e9)) {
            h->n = 0;  // level 0 of a large and nearly empty box
            return;
        }
        g.ncell = (int64_t)cells;
        h->n = l + 1;
        h->first[l + 1] = (int32_t)total;
    }
}

static dcpse_status support_pass(dcpse_ctx* ctx, int dim, const double* pos_sup, int64_t n_sup,
                                 const double* pos_dom, int64_t n_dom, const int32_t* dom_self,
                                 const double* rcut, int rcut_pp,
                                 const double* box_lo, const double* box_hi, unsigned periodic,
                                 int64_t* row_ptr, int32_t* col, int64_t* nnz_out,
                                 const double* rcut_host = nullptr, bool continues = false) {
    if (dim != 2 && dim != 3) return fail(ctx, DCPSE_ERR_UNSUPPORTED, "dim must be 2 or 3");
    // positions of an empty set may be null (a particle set without storage)
    if ((!pos_sup && n_sup > 0) || !row_ptr || !box_lo || !box_hi || n_sup < 0 || n_dom < 0)
        return fail(ctx, DCPSE_ERR_INVALID, "null pointer or negative size");
    if (n_sup >= (int64_t)1 << 31 || n_dom >= (int64_t)1 << 31)
        return fail(ctx, DCPSE_ERR_RANGE, "particle counts must be < 2^31");
    const int same = pos_dom == nullptr;
    // a NULL domain is the support set itself: its row count is n_sup (a
    // smaller n_dom would size row_ptr for fewer rows than are written)
    if (same && n_dom != n_sup)
        return fail(ctx, DCPSE_ERR_INVALID, "pos_dom NULL (the support set as domain) needs n_dom == n_sup");
    if (same) pos_dom = pos_sup;
    // empty sets: no rows, or rows without neighbours
    if (n_dom == 0 || n_sup == 0) {
        if (!col) {  // count pass: row_ptr = 0, nnz = 0
            fill_i64(ctx->stream, row_ptr, n_dom + 1, 0);
            DCPSE_LAUNCH_CHECK(ctx);
            if (nnz_out) *nnz_out = 0;
        }
        return DCPSE_OK;
    }
    if (!rcut) return fail(ctx, DCPSE_ERR_INVALID, "rcut is null");
    hipStream_t s = ctx->stream;
    // the largest cut-off fixes the cell edge
    double rmax = 0.0, rmin = 0.0;
    dcpse_support_cache& sc = ctx->sup;
    if (rcut_host && !rcut_pp) {
        rmin = rmax = *rcut_host;
    } else if (continues && sc.seen && sc.seen_pos == pos_sup && sc.seen_rcut == rcut && sc.seen_n == n_dom) {
        rmax = sc.seen_max;
        rmin = sc.seen_min;
    } else if (rcut_pp) {
        // reduced on the device; only the blocks' extremes come back
        Workspace w0;
        dcpse_status st0 = reserve_workspace(ctx, kMinMaxBlocks * 2 * sizeof(double) + 256, &w0);
        if (st0) return st0;
        double* mm = w0.take<double>(2 * kMinMaxBlocks);
        if (!mm) return fail(ctx, DCPSE_ERR_INVALID, "workspace sizing error");
        const int nb = (int)std::min<int64_t>(kMinMaxBlocks, (n_dom + kMinMaxThreads - 1) / kMinMaxThreads);
        k_minmax<<<nb, kMinMaxThreads, 0, s>>>(rcut, n_dom, mm);
        DCPSE_LAUNCH_CHECK(ctx);
        double hv[2 * kMinMaxBlocks];
        DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(hv, mm, 2 * nb * sizeof(double), hipMemcpyDeviceToHost, s));
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(s));
        rmin = hv[0];
        for (int b = 0; b < nb; ++b) {
            rmin = std::fmin(rmin, hv[2 * b]);
            rmax = std::fmax(rmax, hv[2 * b + 1]);
        }
    } else {
        DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(&rmax, rcut, sizeof(double), hipMemcpyDeviceToHost, s));
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(s));
        rmin = rmax;
    }
    sc.seen = col == nullptr;
    sc.seen_pos = pos_sup;
    sc.seen_rcut = rcut;
    sc.seen_n = n_dom;
    sc.seen_max = rmax;
    sc.seen_min = rmin;
    const double spread = rmin > 0.0 ? rmax / rmin : 1.0;
    CellGrid g;
    HomeLevels home;
    home.n = 0;
    dcpse_status st;
    // One particle set goes by groups (k_group_pairs) where FP32 resolves the
    // pairs (see kPairTol, relative()) and the candidates of a group leave room
    // to sort them in registers; everything else a wavefront per particle.
    bool grouped = same && rmax > 1e-30 && rmax < 1e30;
    for (int d = 0; d < dim; ++d)
        grouped = grouped && std::fabs(box_lo[d]) <= kMaxOffset * rmax && std::fabs(box_hi[d]) <= kMaxOffset * rmax;
    int nws = 0;  // words of a take mask
    if (grouped && !rcut_pp) {
        // cells of edge >= rcut
        if ((st = make_grid(ctx, dim, box_lo, box_hi, periodic, rmax, 1, &g))) return st;
        const double cand = (double)n_sup * (dim == 3 ? 27.0 : 9.0) / (double)g.ncell;
        grouped = cand <= (dim == 3 ? 1638.0 : 819.0);
        // about half of the 3^dim cells' particles are within reach of the
        // cell's own; lists of 0.84 of them leave room for uneven cells
        nws = std::max(2, std::min(32, (int)std::ceil(0.84 * cand / kWave)));
        for (int d = 0; d < dim; ++d)
            grouped = grouped && g.cs[d] <= 0.5 * kMaxReach * rmax && (g.nc[d] >= 4 || !((periodic >> d) & 1u));
    } else if (grouped) {
        // candidate cells of about half the smallest cut-off, at most a few
        // per particle: coarser ones bring more candidates that the box test
        // drops, finer ones more empty cells
        make_levels(dim, box_lo, box_hi, periodic, rmin, rmax, n_sup, &home);
        grouped = home.n > 0 && rmin > 0.0;
        for (int d = 0; d < dim; ++d)
            if ((periodic >> d) & 1u) grouped = grouped && box_hi[d] - box_lo[d] > (kHomeEdge + 2.1) * rmax;
        int K = (int)std::min(dim == 3 ? 8.0 : 16.0, std::ceil(2.0 * spread - 1e-9));
        for (; grouped; --K) {
            // (one cell per cut-off needs three cut-offs of a periodic
            // dimension, the scans of a wavefront per particle 2.5)
            grouped = make_grid(ctx, dim, box_lo, box_hi, periodic, rmax, K, &g) == DCPSE_OK;
            if (!grouped || g.ncell <= 8 * n_sup + 4096 || K == 1) break;
        }
        nws = dim == 3 ? 8 : 4;
    }
    if (!grouped) {
        // cells per cut-off: 2 (3D) or 4 (2D) for one cut-off; with a spread of
        // cut-offs, about rmax / rmin so the smallest scan only their own
        // neighbourhood (bounded: a wave handles 32 cell rows per round)
        const int K = dim == 3 ? std::min(4, std::max(2, (int)std::ceil(spread - 1e-9)))
                               : std::min(8, std::max(4, (int)std::ceil(spread - 1e-9)));
        if ((st = make_grid(ctx, dim, box_lo, box_hi, periodic, rmax, K, &g))) return st;
    }
    const bool pp = grouped && rcut_pp;
    // home cells: the candidate cells, or the levels' cells
    const int64_t n_home = pp ? home.first[home.n] : g.ncell;
    // groups numbered over the occupied home cells where most are empty
    const bool compact = grouped && (pp || n_home > 2 * n_sup);
    const int64_t max_groups = !compact ? n_home : pp ? std::min(n_sup, n_sup / 4 + 4096) : n_sup;

    // the fill of one set reuses the cell list, candidate lists and take masks
    // of the count just before it when the arguments match; with a cut-off per
    // particle, whose values the key does not hold, only where the caller says
    // that they are the count's
    const bool count_pass = col == nullptr;
    const bool cached = grouped && !count_pass && sc.valid && sc.dim == dim && sc.pos == pos_sup &&
                        sc.n == n_sup && sc.rcut == rmax && sc.rmin == rmin && sc.rcut_pp == rcut_pp &&
                        (!rcut_pp || (continues && sc.rcuts == rcut)) &&
                        sc.periodic == periodic && sc.nws == nws &&
                        std::equal(box_lo, box_lo + dim, sc.lo) && std::equal(box_hi, box_hi + dim, sc.hi);
    sc.valid = false;

    // Cell list, candidate lists, masks and the list of particles left to
    // k_support_rows: in the context's support cache when grouped (a fill
    // finds them there), the cell list alone in the workspace otherwise.
    int64_t *cell_start = nullptr, *home_start = nullptr, *group_index = nullptr;
    CellRec *rec = nullptr, *home_rec = nullptr;
    int32_t *group_cell = nullptr, *ncand = nullptr, *lists = nullptr, *spill = nullptr;
    uint64_t* masks = nullptr;
    auto carve_cells = [&](Workspace& cw) {
        cell_start = cw.take<int64_t>(g.ncell + 1);
        rec = cw.take<CellRec>(n_sup);
    };
    auto carve = [&](Workspace& cw) {
        carve_cells(cw);
        home_start = pp ? cw.take<int64_t>(n_home + 1) : cell_start;
        home_rec = pp ? cw.take<CellRec>(n_sup) : rec;
        if (compact) {
            group_index = cw.take<int64_t>(n_home + 1);
            group_cell = cw.take<int32_t>(std::min(n_home, n_sup) + 1);
        }
        masks = cw.take<uint64_t>((size_t)n_sup * nws);
        ncand = cw.take<int32_t>(max_groups + 1);
        lists = cw.take<int32_t>((size_t)max_groups * nws * kWave);
        spill = cw.take<int32_t>(n_sup + 2);
    };
    bool groups_on = grouped && (count_pass || cached);
    if (groups_on) {
        Workspace cw;
        cw.cap = ~size_t(0) >> 1;
        carve(cw);  // sizes only
        const size_t cap = cw.used;
        if (count_pass && sc.cap < cap) {
            DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(s));
            if (sc.buf) (void)hipFree(sc.buf);
            sc.buf = nullptr;
            sc.cap = 0;
            if (hipMalloc(&sc.buf, cap) == hipSuccess) {
                sc.cap = cap;
            } else {
                // no room for the lists: count from positions, and the fill
                // (finding no matching cache) fills from positions too
                (void)hipGetLastError();
                sc.buf = nullptr;
                groups_on = false;
            }
        }
        if (groups_on) {
            cw = Workspace();
            cw.base = static_cast<char*>(sc.buf);
            cw.cap = sc.cap;
            carve(cw);
            if (!spill) return fail(ctx, DCPSE_ERR_INVALID, "support cache sizing error");
        }
    }
    const bool home_on = groups_on && pp;
    Workspace w;
    const size_t need = (size_t)n_sup * 4 * 4 + (size_t)g.ncell * 4 + (size_t)n_home * 8 + (size_t)n_dom * 4 +
                        (groups_on ? 0 : (size_t)(g.ncell + 1) * 8 + (size_t)n_sup * sizeof(CellRec)) +
                        scan_workspace_bytes(std::max(std::max(g.ncell, n_home), n_dom)) + 64 * 256;
    if ((st = reserve_workspace(ctx, need, &w))) return st;
    if (!groups_on) carve_cells(w);
    int32_t* cell_id = w.take<int32_t>(n_sup + 1);
    int32_t* rank = w.take<int32_t>(n_sup + 1);
    int32_t* cell_cnt = w.take<int32_t>(g.ncell + 1);
    int32_t *home_id = nullptr, *home_rank = nullptr, *home_cnt = cell_cnt, *occupied = nullptr;
    if (home_on) {
        home_id = w.take<int32_t>(n_sup + 1);
        home_rank = w.take<int32_t>(n_sup + 1);
        home_cnt = w.take<int32_t>(n_home + 1);
    }
    if (groups_on && compact) occupied = w.take<int32_t>(n_home + 1);
    int32_t* counts = w.take<int32_t>(n_dom + 1);
    int32_t* flags = w.take<int32_t>(64);
    const Workspace ws_scan = w;
    if (!flags) return fail(ctx, DCPSE_ERR_INVALID, "workspace sizing error");

    auto blocks_for = [](int64_t n) {
        return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 16384));
    };
    auto scan = [&](const int32_t* in, int64_t n, int64_t* out) {
        Workspace ws = ws_scan;
        return scan_counts(ctx, in, n, out, &ws);
    };
    const ClearRanges zero = {{flags, cell_cnt, home_cnt, spill},
                              {64, cached ? 0 : g.ncell + 1, home_on && !cached ? n_home + 1 : 0,
                               count_pass && groups_on ? 1 : 0}};
    k_clear<<<blocks_for(std::max<int64_t>(64, cached ? 0 : std::max(g.ncell, home_on ? n_home : 0))), 256, 0, s>>>(zero);
    DCPSE_LAUNCH_CHECK(ctx);
    if (!cached) {
        const unsigned tb = blocks_for(n_sup);
        auto cells = [&](auto D, auto H) {
            constexpr int DIM = decltype(D)::value;
            constexpr bool HOME = decltype(H)::value;
            k_cell_assign<DIM, HOME><<<tb, 256, 0, s>>>(pos_sup, n_sup, rcut, g, home, cell_id, rank, cell_cnt,
                                                       home_id, home_rank, home_cnt);
            DCPSE_LAUNCH_CHECK(ctx);
            dcpse_status sst;
            if ((sst = scan(cell_cnt, g.ncell, cell_start))) return sst;
            if (HOME && (sst = scan(home_cnt, n_home, home_start))) return sst;
            k_cell_fill<DIM, HOME><<<tb, 256, 0, s>>>(pos_sup, n_sup, cell_id, rank, cell_start, rec, home_id,
                                                     home_rank, home_start, home_rec);
            DCPSE_LAUNCH_CHECK(ctx);
            return DCPSE_OK;
        };
        auto by_home = [&](auto D) { return home_on ? cells(D, std::true_type()) : cells(D, std::false_type()); };
        st = dim == 2 ? by_home(std::integral_constant<int, 2>()) : by_home(std::integral_constant<int, 3>());
        if (st) return st;
        if (occupied) {
            k_occupied<<<blocks_for(n_home), 256, 0, s>>>(home_cnt, n_home, occupied);
            DCPSE_LAUNCH_CHECK(ctx);
            if ((st = scan(occupied, n_home, group_index))) return st;
            k_group_cells<<<blocks_for(n_home), 256, 0, s>>>(home_cnt, group_index, n_home, group_cell);
            DCPSE_LAUNCH_CHECK(ctx);
        }
    }
    Groups a;
    a.n = n_sup;
    a.pos = pos_sup;
    a.rcut = rcut;
    a.g = g;
    a.cell_start = cell_start;
    a.rec = rec;
    a.home_start = home_start;
    a.home = home_rec;
    a.group_cell = group_cell;
    a.n_groups = group_cell ? group_index + n_home : nullptr;
    a.max_groups = max_groups;
    a.counts = counts;
    a.flags = flags;
    a.ncand = ncand;
    a.lists = lists;
    a.masks = masks;
    a.nws = nws;
    a.spill = spill;
    // a wavefront per group, the blocks in whole rounds over the XCDs
    const int64_t launch_groups_n = compact ? std::min(n_home, n_sup) : n_home;
    const unsigned group_blocks = (unsigned)((launch_groups_n + kPairWaves * 8 - 1) / (kPairWaves * 8) * 8);
    const unsigned row_blocks = (unsigned)std::max<int64_t>(
        1, std::min<int64_t>((n_dom + kRowWaves - 1) / kRowWaves, (int64_t)ctx->num_cus * 16));
    // every row (list NULL) or the listed ones from positions
    auto rows = [&](auto F, const int32_t* list) {
        constexpr bool FILL = decltype(F)::value;
        if (dim == 2)
            k_support_rows<2, FILL><<<row_blocks, kRowWaves * kWave, 0, s>>>(
                pos_dom, n_dom, same, dom_self, rcut, rcut_pp, g, cell_start, rec, counts, flags, row_ptr, col, list);
        else
            k_support_rows<3, FILL><<<row_blocks, kRowWaves * kWave, 0, s>>>(
                pos_dom, n_dom, same, dom_self, rcut, rcut_pp, g, cell_start, rec, counts, flags, row_ptr, col, list);
    };
    if (count_pass) {
        if (groups_on) {
            // candidate lists and masks, then the particles they do not cover
            launch_groups(dim, nws, [&](auto D, auto R) {
                constexpr int DIM = decltype(D)::value, RM = decltype(R)::value;
                if (pp) k_group_pairs<DIM, RM, true><<<group_blocks, kPairWaves * kWave, 0, s>>>(a, home);
                else k_group_pairs<DIM, RM, false><<<group_blocks, kPairWaves * kWave, 0, s>>>(a, home);
            });
            DCPSE_LAUNCH_CHECK(ctx);
            rows(std::false_type(), spill);
        } else {
            rows(std::false_type(), nullptr);
        }
        DCPSE_LAUNCH_CHECK(ctx);
        {
            Workspace ws = ws_scan;
            if ((st = scan_counts(ctx, counts, n_dom, row_ptr, &ws, true, flags, groups_on ? spill : nullptr))) return st;
        }
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(s));
        const int64_t nnz = ctx->host[0];
        const int32_t ovf = (int32_t)ctx->host[1], n_spill = groups_on ? (int32_t)ctx->host[2] : 0;
        if (ovf & 1)
            return fail(ctx, DCPSE_ERR_RANGE, "a support row exceeds DCPSE_MAX_ROW=%d neighbours",
                        DCPSE_MAX_ROW);
        if (nnz >= ((int64_t)1 << 31) * 64)
            return fail(ctx, DCPSE_ERR_RANGE, "nnz out of range");
        if (nnz_out) *nnz_out = nnz;
        if (groups_on) {
            sc.valid = true;
            sc.spill = n_spill > 0;
            sc.dim = dim;
            sc.pos = pos_sup;
            sc.n = n_sup;
            sc.rcut = rmax;
            sc.rmin = rmin;
            sc.rcut_pp = rcut_pp;
            sc.rcuts = rcut;
            sc.periodic = periodic;
            sc.nws = nws;
            for (int d = 0; d < 3; ++d) {
                sc.lo[d] = d < dim ? box_lo[d] : 0.0;
                sc.hi[d] = d < dim ? box_hi[d] : 0.0;
            }
        }
    } else {
        if (cached) {
            launch_groups(dim, nws, [&](auto, auto R) {
                k_group_rows<decltype(R)::value><<<group_blocks, kPairWaves * kWave, 0, s>>>(a, row_ptr, col);
            });
            DCPSE_LAUNCH_CHECK(ctx);
        }
        if (!cached || sc.spill) {
            rows(std::true_type(), cached ? spill : nullptr);
            DCPSE_LAUNCH_CHECK(ctx);
            const int64_t lb = std::max<int64_t>(
                1, std::min<int64_t>((n_dom + kRowWaves * kWave - 1) / (kRowWaves * kWave), (int64_t)ctx->num_cus * 8));
            k_sort_long_rows<<<(unsigned)lb, kRowWaves * kWave, 0, s>>>(n_dom, row_ptr, col);
            DCPSE_LAUNCH_CHECK(ctx);
        }
        k_to_host<<<1, 1, 0, s>>>(flags, ctx->host);
        DCPSE_LAUNCH_CHECK(ctx);
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(s));
        const int32_t ovf = (int32_t)ctx->host[0];
        if (sc.cap > sc.keep) {  // a large set's lists are not kept (25M particles and more)
            (void)hipFree(sc.buf);
            sc.buf = nullptr;
            sc.cap = 0;
        }
        if (ovf & 3)
            return fail(ctx, DCPSE_ERR_INVALID,
                        "support fill disagrees with row_ptr (positions or rcut changed since count?)");
    }
    return DCPSE_OK;
}

// ---------------------------------------------------------------------------
// transposed CSR
// ---------------------------------------------------------------------------
__global__ void k_tcount(const int32_t* __restrict__ col, int64_t nnz, int32_t* __restrict__ cnt) {
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < nnz;
         j += (int64_t)gridDim.x * blockDim.x)
        atomicAdd(&cnt[col[j]], 1);
}

// One wavefront per source row p, a lane per entry: each entry takes its
// slot in transposed row col[j] by an atomic cursor (the order is undone by
// k_tsort) and the row sum for diag[p] is a wave sum in FP64.
template <typename T>
__global__ __launch_bounds__(kRowWaves * kWave) void k_tfill(int64_t n_rows, const int64_t* __restrict__ row_ptr,
                                                             const int32_t* __restrict__ col,
                                                             const T* __restrict__ W,
                                                             const int64_t* __restrict__ rowT_ptr,
                                                             int32_t* __restrict__ cursor,
                                                             int32_t* __restrict__ colT, T* __restrict__ WT,
                                                             T* __restrict__ diag) {
    const int lane = threadIdx.x & 63;
    for (int64_t p = (int64_t)blockIdx.x * kRowWaves + (threadIdx.x >> 6); p < n_rows;
         p += (int64_t)gridDim.x * kRowWaves) {
        const int64_t rs = row_ptr[p], re = row_ptr[p + 1];
        double acc = 0.0;
        for (int64_t j = rs + lane; j < re; j += kWave) {
            const int32_t q = col[j];
            const T wj = W[j];
            const int64_t at = rowT_ptr[q] + atomicAdd(&cursor[q], 1);
            colT[at] = (int32_t)p;
            WT[at] = wj;
            acc += (double)wj;
        }
        acc = wave_sum(acc);
        if (lane == 0) diag[p] = (T)(-acc);
    }
}

// Transpose of a structurally symmetric CSR with strictly ascending rows (a
// support of one set with one cut-off): the transpose has the same row_ptr
// and col, and its entry k = (q, p) of row q takes the weight of entry (p, q),
// found by searching q in row p. One wavefront per output row q, a lane per
// entry, so the writes are coalesced and there are no atomics and no sort.
// The search starts at the mirror position len_p - 1 - m (exact for a
// lattice stencil, m = index of p in row q), then bisects. Raises *asym,
// leaving the outputs to the general path, when a row is not strictly
// ascending, when a transposed length differs, or when q is missing from
// row p; each row checks its own entries, so both directions of every pair
// are covered.
template <typename T>
__global__ __launch_bounds__(kRowWaves * kWave) void k_tfill_sym(int64_t n_rows, const int64_t* __restrict__ row_ptr,
                                                                 const int32_t* __restrict__ col,
                                                                 const T* __restrict__ W,
                                                                 const int64_t* __restrict__ rowT_ptr,
                                                                 int32_t* __restrict__ colT, T* __restrict__ WT,
                                                                 T* __restrict__ diag, int32_t* __restrict__ asym) {
    const int lane = threadIdx.x & 63;
    // consecutive logical blocks on one XCD (blocks are dealt round-robin over
    // the 8 XCDs): the rows searched by neighbouring rows q share cache lines
    const unsigned G = gridDim.x;
    const unsigned lb = (G % 8u == 0u) ? (blockIdx.x % 8u) * (G / 8u) + blockIdx.x / 8u : blockIdx.x;
    for (int64_t q = (int64_t)lb * kRowWaves + (threadIdx.x >> 6); q < n_rows; q += (int64_t)G * kRowWaves) {
        const int64_t rs = row_ptr[q], re = row_ptr[q + 1];
        bool bad = lane == 0 && (rowT_ptr[q] != rs || (q + 1 == n_rows && rowT_ptr[n_rows] != re));
        double acc = 0.0;
        for (int64_t k = rs + lane; k < re; k += kWave) {
            const int32_t p = col[k];
            acc += (double)W[k];
            colT[k] = p;
            if (k + 1 < re && col[k + 1] <= p) bad = true;
            if (p < 0 || p >= n_rows) {
                bad = true;
                continue;
            }
            const int64_t ps = row_ptr[p], pe = row_ptr[p + 1];
            const int64_t mirror = pe - 1 - (k - rs);
            int64_t lo = ps, hi = pe;
            if (mirror >= ps && mirror < pe) {
                const int32_t c = col[mirror];
                if (c == (int32_t)q) lo = hi = mirror;
                else if (c < (int32_t)q) lo = mirror + 1;
                else hi = mirror;
            }
            // first position in [lo, hi) with col >= q
            while (lo < hi) {
                const int64_t mid = lo + ((hi - lo) >> 1);
                if (col[mid] < (int32_t)q) lo = mid + 1;
                else hi = mid;
            }
            if (lo < pe && col[lo] == (int32_t)q) WT[k] = W[lo];
            else bad = true;
        }
        acc = wave_sum(acc);
        if (lane == 0) diag[q] = (T)(-acc);
        if (__ballot(bad) && lane == 0) atomicOr(asym, 1);
    }
}

// Sorts each transposed row by ascending source row (rank sort in LDS); rows
// longer than DCPSE_MAX_ROW raise *overflow and are left unsorted.
template <typename T>
__global__ __launch_bounds__(kRowWaves * kWave) void k_tsort(int64_t n_cols, const int64_t* __restrict__ rowT_ptr,
                                                             int32_t* __restrict__ colT, T* __restrict__ WT,
                                                             int32_t* __restrict__ overflow) {
    __shared__ int32_t kbuf[kRowWaves][DCPSE_MAX_ROW];
    __shared__ T vbuf[kRowWaves][DCPSE_MAX_ROW];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    for (int64_t r = (int64_t)blockIdx.x * kRowWaves + wv; r < n_cols; r += (int64_t)gridDim.x * kRowWaves) {
        const int64_t rs = rowT_ptr[r];
        const int64_t n64 = rowT_ptr[r + 1] - rs;
        if (n64 > DCPSE_MAX_ROW) {
            if (lane == 0) atomicOr(overflow, 1);
            continue;
        }
        const int n = (int)n64;
        for (int e = lane; e < n; e += kWave) {
            kbuf[wv][e] = colT[rs + e];
            vbuf[wv][e] = WT[rs + e];
        }
        wave_lds_sync();
        for (int e = lane; e < n; e += kWave) {
            const int key = kbuf[wv][e];
            int rank = 0;
            for (int j = 0; j < n; ++j) rank += kbuf[wv][j] < key;
            colT[rs + rank] = key;
            WT[rs + rank] = vbuf[wv][e];
        }
        wave_lds_sync();
    }
}

template <typename T>
static dcpse_status transpose_fill(dcpse_ctx* ctx, int64_t n_rows, int64_t n_cols, const int64_t* row_ptr,
                                   const int32_t* col, const T* W, const int64_t* rowT_ptr, int32_t* colT,
                                   T* WT, T* diag) {
    if (!row_ptr || !col || !W || !rowT_ptr || !colT || !WT || !diag || n_rows < 0 || n_cols < 0)
        return fail(ctx, DCPSE_ERR_INVALID, "null pointer or negative size");
    if (n_rows != n_cols)
        return fail(ctx, DCPSE_ERR_UNSUPPORTED, "transpose needs the domain set to be the support set");
    Workspace w;
    dcpse_status st = reserve_workspace(ctx, (size_t)(n_cols + 64) * 4 + 1024, &w);
    if (st) return st;
    int32_t* cursor = w.take<int32_t>(n_cols + 1);
    int32_t* flags = w.take<int32_t>(16);
    hipStream_t s = ctx->stream;
    fill_i32(s, cursor, n_cols + 1, 0);
    fill_i32(s, flags, 16, 0);
    if (n_rows > 0) {
        int64_t b = std::max<int64_t>(1, std::min<int64_t>((n_rows + kRowWaves - 1) / kRowWaves,
                                                           (int64_t)ctx->num_cus * 32));
        // a symmetric pattern with sorted rows first; the general path below
        // only if it reports otherwise
        const unsigned bs = (unsigned)(b >= 8 ? b / 8 * 8 : b);
        k_tfill_sym<T><<<bs, kRowWaves * kWave, 0, s>>>(n_rows, row_ptr, col, W, rowT_ptr, colT, WT, diag, flags + 1);
        DCPSE_LAUNCH_CHECK(ctx);
        int32_t asym = 0;
        DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(&asym, flags + 1, sizeof(int32_t), hipMemcpyDeviceToHost, s));
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(s));
        if (!asym) return DCPSE_OK;
        k_tfill<T><<<(unsigned)b, kRowWaves * kWave, 0, s>>>(n_rows, row_ptr, col, W, rowT_ptr, cursor, colT, WT,
                                                              diag);
        DCPSE_LAUNCH_CHECK(ctx);
        int64_t rb = std::max<int64_t>(1, std::min<int64_t>((n_cols + kRowWaves - 1) / kRowWaves,
                                                            (int64_t)ctx->num_cus * 16));
        k_tsort<T><<<(unsigned)rb, kRowWaves * kWave, 0, s>>>(n_cols, rowT_ptr, colT, WT, flags);
        DCPSE_LAUNCH_CHECK(ctx);
    }
    int32_t ovf = 0;
    DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(&ovf, flags, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(s));
    if (ovf) return fail(ctx, DCPSE_ERR_RANGE, "a transposed row exceeds DCPSE_MAX_ROW=%d", DCPSE_MAX_ROW);
    return DCPSE_OK;
}

}  // namespace dcpse

using namespace dcpse;

extern "C" {

dcpse_status dcpse_support_count(dcpse_ctx* ctx, int32_t dim, const double* pos_sup, int64_t n_sup,
                                 const double* pos_dom, int64_t n_dom, const double* rcut,
                                 int32_t rcut_per_particle, const double* box_lo, const double* box_hi,
                                 uint32_t periodic_mask, int64_t* row_ptr, int64_t* nnz) {
    if (!ctx) return DCPSE_ERR_INVALID;
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    return support_pass(ctx, dim, pos_sup, n_sup, pos_dom, n_dom, nullptr, rcut, rcut_per_particle, box_lo, box_hi,
                        periodic_mask, row_ptr, nullptr, nnz);
}

dcpse_status dcpse_support_fill(dcpse_ctx* ctx, int32_t dim, const double* pos_sup, int64_t n_sup,
                                const double* pos_dom, int64_t n_dom, const double* rcut,
                                int32_t rcut_per_particle, const double* box_lo, const double* box_hi,
                                uint32_t periodic_mask, const int64_t* row_ptr, int32_t* col) {
    if (!ctx) return DCPSE_ERR_INVALID;
    if (!col) return fail(ctx, DCPSE_ERR_INVALID, "col is null");
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    return support_pass(ctx, dim, pos_sup, n_sup, pos_dom, n_dom, nullptr, rcut, rcut_per_particle, box_lo, box_hi,
                        periodic_mask, const_cast<int64_t*>(row_ptr), col, nullptr);
}

dcpse_status dcpse_support_count_subset(dcpse_ctx* ctx, int32_t dim, const double* pos_sup, int64_t n_sup,
                                        const double* pos_dom, const int32_t* dom_ids, int64_t n_dom,
                                        const double* rcut, int32_t rcut_per_particle, const double* box_lo,
                                        const double* box_hi, uint32_t periodic_mask, int64_t* row_ptr,
                                        int64_t* nnz) {
    if (!ctx) return DCPSE_ERR_INVALID;
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    if (n_dom == 0 && row_ptr) {  // an empty subset: no rows
        fill_i64(ctx->stream, row_ptr, 1, 0);
        DCPSE_LAUNCH_CHECK(ctx);
        if (nnz) *nnz = 0;
        return DCPSE_OK;
    }
    if (!pos_dom || !dom_ids) return fail(ctx, DCPSE_ERR_INVALID, "a subset needs pos_dom and dom_ids");
    return support_pass(ctx, dim, pos_sup, n_sup, pos_dom, n_dom, dom_ids, rcut, rcut_per_particle, box_lo, box_hi,
                        periodic_mask, row_ptr, nullptr, nnz);
}

dcpse_status dcpse_support_fill_subset(dcpse_ctx* ctx, int32_t dim, const double* pos_sup, int64_t n_sup,
                                       const double* pos_dom, const int32_t* dom_ids, int64_t n_dom,
                                       const double* rcut, int32_t rcut_per_particle, const double* box_lo,
                                       const double* box_hi, uint32_t periodic_mask, const int64_t* row_ptr,
                                       int32_t* col) {
    if (!ctx) return DCPSE_ERR_INVALID;
    if (n_dom == 0) return DCPSE_OK;  // an empty subset: no rows
    if (!col) return fail(ctx, DCPSE_ERR_INVALID, "col is null");
    if (!pos_dom || !dom_ids) return fail(ctx, DCPSE_ERR_INVALID, "a subset needs pos_dom and dom_ids");
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    return support_pass(ctx, dim, pos_sup, n_sup, pos_dom, n_dom, dom_ids, rcut, rcut_per_particle, box_lo, box_hi,
                        periodic_mask, const_cast<int64_t*>(row_ptr), col, nullptr);
}

dcpse_status dcpse_support_count_one(dcpse_ctx* ctx, int32_t dim, const double* pos_sup, int64_t n_sup,
                                     const double* pos_dom, const int32_t* dom_ids, int64_t n_dom, const double* rcut,
                                     double rcut_value, const double* box_lo, const double* box_hi,
                                     uint32_t periodic_mask, int64_t* row_ptr, int64_t* nnz) {
    if (!ctx) return DCPSE_ERR_INVALID;
    if (dom_ids && !pos_dom) return fail(ctx, DCPSE_ERR_INVALID, "a subset needs pos_dom and dom_ids");
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    return support_pass(ctx, dim, pos_sup, n_sup, pos_dom, n_dom, dom_ids, rcut, 0, box_lo, box_hi, periodic_mask,
                        row_ptr, nullptr, nnz, &rcut_value);
}

dcpse_status dcpse_support_fill_counted(dcpse_ctx* ctx, int32_t dim, const double* pos_sup, int64_t n_sup,
                                        const double* pos_dom, const int32_t* dom_ids, int64_t n_dom,
                                        const double* rcut, int32_t rcut_per_particle, const double* box_lo,
                                        const double* box_hi, uint32_t periodic_mask, const int64_t* row_ptr,
                                        int32_t* col) {
    if (!ctx) return DCPSE_ERR_INVALID;
    if (!col) return fail(ctx, DCPSE_ERR_INVALID, "col is null");
    if (dom_ids && !pos_dom) return fail(ctx, DCPSE_ERR_INVALID, "a subset needs pos_dom and dom_ids");
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    return support_pass(ctx, dim, pos_sup, n_sup, pos_dom, n_dom, dom_ids, rcut, rcut_per_particle, box_lo, box_hi,
                        periodic_mask, const_cast<int64_t*>(row_ptr), col, nullptr, nullptr, true);
}

dcpse_status dcpse_transpose_count(dcpse_ctx* ctx, int64_t n_rows, int64_t n_cols, const int64_t* row_ptr,
                                   const int32_t* col, int64_t* rowT_ptr) {
    if (!ctx) return DCPSE_ERR_INVALID;
    if (!row_ptr || !col || !rowT_ptr || n_rows < 0 || n_cols < 0)
        return fail(ctx, DCPSE_ERR_INVALID, "null pointer or negative size");
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    int64_t nnz = 0;
    DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(&nnz, row_ptr + n_rows, sizeof(int64_t), hipMemcpyDeviceToHost, ctx->stream));
    DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
    Workspace w;
    dcpse_status st = reserve_workspace(ctx, (size_t)(n_cols + 1) * 4 + scan_workspace_bytes(n_cols) + 1024, &w);
    if (st) return st;
    const WorkspaceUse use(ctx);
    int32_t* cnt = w.take<int32_t>(n_cols + 1);
    fill_i32(ctx->stream, cnt, n_cols + 1, 0);
    if (nnz > 0) {
        int64_t b = std::max<int64_t>(1, std::min<int64_t>((nnz + 255) / 256, 65536));
        k_tcount<<<(unsigned)b, 256, 0, ctx->stream>>>(col, nnz, cnt);
        DCPSE_LAUNCH_CHECK(ctx);
    }
    return scan_counts(ctx, cnt, n_cols, rowT_ptr, &w);
}

dcpse_status dcpse_transpose_fill_f32(dcpse_ctx* ctx, int64_t n_rows, int64_t n_cols, const int64_t* row_ptr,
                                      const int32_t* col, const float* W, const int64_t* rowT_ptr,
                                      int32_t* colT, float* WT, float* diag) {
    if (!ctx) return DCPSE_ERR_INVALID;
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    return transpose_fill<float>(ctx, n_rows, n_cols, row_ptr, col, W, rowT_ptr, colT, WT, diag);
}

dcpse_status dcpse_transpose_fill_f64(dcpse_ctx* ctx, int64_t n_rows, int64_t n_cols, const int64_t* row_ptr,
                                      const int32_t* col, const double* W, const int64_t* rowT_ptr,
                                      int32_t* colT, double* WT, double* diag) {
    if (!ctx) return DCPSE_ERR_INVALID;
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    return transpose_fill<double>(ctx, n_rows, n_cols, row_ptr, col, W, rowT_ptr, colT, WT, diag);
}

}  // extern "C"
