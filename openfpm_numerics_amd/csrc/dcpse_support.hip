// Neighbour-support (Verlet CSR) builder, device scan and transposed-CSR
// builder for gfx950.
//
// Support semantics follow the reference's Verlet list for DC-PSE
// (VL_NON_SYMMETRIC | VL_SKIP_REF_PART: q != p, |x_p - x_q| < rCut), see
// src/DCPSE/SupportBuilder.cuh:15-61. Unlike that builder (one thread per
// particle, host-side serial prefix sum, size_t keys, 4 host round trips), the
// whole CSR is built on the device: a cell grid by counting sort, then one
// wavefront per cell (one set, one cut-off) or per particle over the
// neighbouring cells' particles, flattened into one candidate list and sorted
// in registers, so every row comes out in ascending particle index
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

__global__ __launch_bounds__(kScanBlock) void k_scan_tiles(const int32_t* __restrict__ in, int64_t n,
                                                           const int64_t* __restrict__ tsum,
                                                           int64_t* __restrict__ out) {
    __shared__ long long buf[kScanBlock];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    long long v[kScanItems];
    long long tot = 0;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        int64_t k = base + i;
        v[i] = k < n ? in[k] : 0;
        tot += v[i];
    }
    buf[threadIdx.x] = tot;
    __syncthreads();
    for (int off = 1; off < kScanBlock; off <<= 1) {
        long long t = threadIdx.x >= (unsigned)off ? buf[threadIdx.x - off] : 0;
        __syncthreads();
        buf[threadIdx.x] += t;
        __syncthreads();
    }
    long long run = tsum[blockIdx.x] + buf[threadIdx.x] - tot;
#pragma unroll
    for (int i = 0; i < kScanItems; ++i) {
        int64_t k = base + i;
        if (k < n) out[k] = run;
        run += v[i];
    }
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = tsum[gridDim.x];
}

size_t scan_workspace_bytes(int64_t n) {
    int64_t nt = (n + kScanTile - 1) / kScanTile;
    return (size_t)(nt + 1) * sizeof(int64_t) + 256;
}

dcpse_status scan_counts(dcpse_ctx* ctx, const int32_t* in, int64_t n, int64_t* out, Workspace* w) {
    int64_t nt = (n + kScanTile - 1) / kScanTile;
    if (nt == 0) nt = 1;
    int64_t* tsum = w->take<int64_t>((size_t)nt + 1);
    if (!tsum) return fail(ctx, DCPSE_ERR_INVALID, "scan: workspace too small");
    k_scan_tilesum<<<(unsigned)nt, kScanBlock, 0, ctx->stream>>>(in, n, tsum);
    DCPSE_LAUNCH_CHECK(ctx);
    k_scan_tilesums<<<1, 1024, 0, ctx->stream>>>(tsum, nt);
    DCPSE_LAUNCH_CHECK(ctx);
    k_scan_tiles<<<(unsigned)nt, kScanBlock, 0, ctx->stream>>>(in, n, tsum, out);
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

dcpse_status reserve_workspace(dcpse_ctx* ctx, size_t bytes, Workspace* w) {
    if (ctx->ws_size < bytes) {
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
        if (ctx->ws) DCPSE_HIP_CHECK(ctx, hipFree(ctx->ws));
        ctx->ws = nullptr;
        size_t nb = std::max(bytes, ctx->ws_size * 2);
        DCPSE_HIP_CHECK(ctx, hipMalloc(&ctx->ws, nb));
        ctx->ws_size = nb;
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

template <int DIM>
__global__ void k_cell_assign(const double* __restrict__ pos, int64_t n, CellGrid g,
                              int32_t* __restrict__ cell_id, int32_t* __restrict__ cell_cnt) {
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n;
         q += (int64_t)gridDim.x * blockDim.x) {
        int64_t c = 0, stride = 1;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            c += stride * cell_of(pos[d * n + q], d, g);
            stride *= g.nc[d];
        }
        cell_id[q] = (int32_t)c;
        atomicAdd(&cell_cnt[c], 1);
    }
}

// cell_part[slot] = particle, and a copy of its position in cell order
// (pos_cell[d * n + slot]) so the row kernels read candidate positions
// contiguously per cell, without waiting for the particle index first.
template <int DIM>
__global__ void k_cell_fill(const int32_t* __restrict__ cell_id, int64_t n, const double* __restrict__ pos,
                            const int64_t* __restrict__ cell_start, int32_t* __restrict__ cursor,
                            int32_t* __restrict__ cell_part, double* __restrict__ pos_cell) {
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n;
         q += (int64_t)gridDim.x * blockDim.x) {
        int32_t c = cell_id[q];
        int64_t at = cell_start[c] + atomicAdd(&cursor[c], 1);
        cell_part[at] = (int32_t)q;
#pragma unroll
        for (int d = 0; d < DIM; ++d) pos_cell[d * n + at] = pos[d * n + q];
    }
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

// One wavefront per domain particle. FILL = false: count the support of p into
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
    const double* __restrict__ pos_sup, int64_t n_sup, const double* __restrict__ pos_dom,
    int64_t n_dom, int same_set, const int32_t* __restrict__ dom_self, const double* __restrict__ rcut, int rcut_pp,
    CellGrid g, const int64_t* __restrict__ cell_start, const int32_t* __restrict__ cell_part,
    const double* __restrict__ pos_cell, int32_t* __restrict__ counts, int32_t* __restrict__ overflow,
    const int64_t* __restrict__ row_ptr, int32_t* __restrict__ col) {
    __shared__ int32_t buf[FILL ? kRowWaves : 1][FILL ? DCPSE_MAX_ROW : 1];
    __shared__ int32_t mark[kRowWaves][kWave];      // segment starting at a candidate of the round
    __shared__ long long seg_cst[kRowWaves][kWave];  // first cell slot of each segment
    __shared__ int32_t seg_ex[kRowWaves][kWave];     // candidates before each segment
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    for (int64_t p = (int64_t)blockIdx.x * kRowWaves + wv; p < n_dom;
         p += (int64_t)gridDim.x * kRowWaves) {
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
                const int q = cell_part[slot];
                double d[3];
#pragma unroll
                for (int dd = 0; dd < DIM; ++dd)
                    d[dd] = min_image_r(xp[dd] - pos_cell[dd * n_sup + slot], g.len[dd], g.ilen[dd],
                                        (g.periodic >> dd) & 1u);
                double d2 = d[DIM - 1] * d[DIM - 1];
#pragma unroll
                for (int dd = DIM - 2; dd >= 0; --dd) d2 = fma(d[dd], d[dd], d2);
                const bool take = (base + lane < total) && q != self_q && d2 < r2;
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

// ---- one set, one cut-off: a wavefront per cell of edge >= rcut -----------
// The candidates of a cell are its 3^dim neighbouring cells, scanned as
// 3^(dim-1) rows along dimension 0 (contiguous in the cell order, split in two
// where a periodic wrap cuts a row), flattened into one list. The count pass
// (k_cell_pairs) keeps the candidates within the cut-off of the bounding box
// of the cell's particles, sorts their indices once per cell, and tests every
// particle of the cell against them: it stores the sorted candidate list of
// the cell and, per particle, which of them it takes (one bit each). The fill
// (k_cell_rows) writes a particle's row as the marked entries of its cell's
// list, which are in ascending order as they stand: no distance work and no
// sort per row. Cells with more candidates than the list holds are left to
// k_support_cells, which tests each particle against positions (restaging
// them per particle when they exceed one LDS copy). All use the distance
// formula of k_support_rows on the same positions (k_cell_pairs wherever FP32
// leaves the outcome open), so the results are the same.
constexpr int kCellWaves = 2;
template <int DIM>
struct CellCap {  // candidates per LDS copy of k_support_cells
    static constexpr int v = DIM == 3 ? 384 : 256;
};

// Block b's cell range: consecutive logical blocks on one XCD (blocks are
// dealt round-robin over the 8 XCDs), so neighbouring cells, which share most
// candidates, meet in one L2.
__device__ __forceinline__ unsigned xcd_block() {
    const unsigned G = gridDim.x;
    return (G % 8u == 0u) ? (blockIdx.x % 8u) * (G / 8u) + blockIdx.x / 8u : blockIdx.x;
}

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
__device__ __forceinline__ void cell_segments(const CellGrid& g, const int64_t* __restrict__ cell_start, int64_t c,
                                              int lane, long long& cst, int& ccnt) {
    int cc[3];
    cell_coords<DIM>(g, c, cc);
    constexpr int ROWS = DIM == 3 ? 9 : 3;
    cst = 0;
    ccnt = 0;
    const int row = lane >> 1, part = lane & 1;
    if (row >= ROWS) return;
    int cy = cc[1] + row % 3 - 1, cz = DIM == 3 ? cc[2] + row / 3 - 1 : 0;
    bool ok = true;
    if ((g.periodic >> 1) & 1u) cy = (cy + g.nc[1]) % g.nc[1];
    else ok &= cy >= 0 && cy < g.nc[1];
    if (DIM == 3) {
        if ((g.periodic >> 2) & 1u) cz = (cz + g.nc[2]) % g.nc[2];
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

// Copies candidates [c0, c0 + cn) of a cell (c0 a multiple of 64) to the
// wave's LDS slice: sq[k - c0] = particle, and with POS its position
// sx[d * sx_stride + k - c0]. A candidate's segment is the last non-empty one
// starting at or before it: the segment starts of each round of 64 are
// marked, a prefix maximum spreads them, and the last one carries over.
// seg_cst / seg_ex (each lane's segment start slot and candidates before it)
// must be written before the call; ends with the slice readable.
template <int DIM, bool POS>
__device__ __forceinline__ void stage_candidates(int c0, int cn, int ccnt, int excl, int32_t* mark,
                                                 const long long* seg_cst, const int32_t* seg_ex,
                                                 const int32_t* __restrict__ cell_part,
                                                 const double* __restrict__ pos_cell, int64_t n, int32_t* sq,
                                                 double* sx, int sx_stride, int lane) {
    int carry = 0;
    for (int base = 0; base < c0 + cn; base += kWave) {
        mark[lane] = -1;
        wave_lds_sync();
        if (ccnt > 0 && excl >= base && excl < base + kWave) mark[excl - base] = lane;
        wave_lds_sync();
        const int seg = max(wave_incl_max(mark[lane]), carry);
        carry = __builtin_amdgcn_readlane(seg, 63);
        const int k = base + lane;
        if (base >= c0 && k < c0 + cn) {
            const int64_t slot = seg_cst[seg] + (k - seg_ex[seg]);
            sq[k - c0] = cell_part[slot];
            if (POS) {
#pragma unroll
                for (int d = 0; d < DIM; ++d) sx[d * sx_stride + k - c0] = pos_cell[d * n + slot];
            }
        }
    }
    wave_lds_sync();
}

// The distance test of a candidate at xq against xp (the minimum image in
// periodic dimensions), as in k_support_rows.
template <int DIM>
__device__ __forceinline__ bool within_cut_at(const double* xp, const double* xq, const CellGrid& g, double r2) {
    double d[3];
#pragma unroll
    for (int dd = 0; dd < DIM; ++dd)
        d[dd] = min_image_r(xp[dd] - xq[dd], g.len[dd], g.ilen[dd], (g.periodic >> dd) & 1u);
    double d2 = d[DIM - 1] * d[DIM - 1];
#pragma unroll
    for (int dd = DIM - 2; dd >= 0; --dd) d2 = fma(d[dd], d[dd], d2);
    return d2 < r2;
}

// ... of candidate slot t of the LDS copy.
template <int DIM>
__device__ __forceinline__ bool within_cut(const double* xp, const double* sx, int sx_stride, int t, const CellGrid& g,
                                           double r2) {
    double xq[3];
#pragma unroll
    for (int dd = 0; dd < DIM; ++dd) xq[dd] = sx[dd * sx_stride + t];
    return within_cut_at<DIM>(xp, xq, g, r2);
}

// Candidates are handled in coordinates relative to the cell centre, in units
// of the cut-off, in FP32: there |a - b|^2 is within 4e-6 of the FP64 value
// for cells up to four cut-offs wide whose positions lie within kMaxOffset
// cut-offs of the origin (FP64 then resolves 1e-9 cut-offs), so outside
// 1 +- kPairTol it decides the pair and inside the FP64 formula does.
constexpr float kPairTol = 2e-5f;
constexpr double kMaxOffset = 1e7;
constexpr int kPairWaves = 4;  // cells (wavefronts) per block

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

// Minimum and maximum over the 64 lanes, in every lane.
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

// What a wave knows of its cell: centre, reciprocal cut-off, particles.
template <int DIM>
struct PairCell {
    double ctr[3];
    double ir;  // 1 / cut-off
    double r2;
    int64_t pst;
    int np, total;  // particles; candidates kept
};

// Position x (component d) relative to the cell centre in units of the
// cut-off: the image nearest to the centre in a periodic dimension. With at
// least four cells per period the candidates' nearest images are the ones the
// pair's minimum image takes wherever the pair is within the cut-off.
template <int DIM>
__device__ __forceinline__ float relative(const PairCell<DIM>& pc, const CellGrid& g, double x, int d) {
    return (float)(min_image_r(x - pc.ctr[d], g.len[d], g.ilen[d], (g.periodic >> d) & 1u) * pc.ir);
}

// Sorts the cell's pc.total <= R * 64 candidate indices (in the wave's LDS
// list), stores them to list[0 ..) and tests the cell's particles against them.
template <int DIM, int R>
__device__ __forceinline__ void pair_tests(const PairCell<DIM>& pc, const CellGrid& g, int64_t n,
                                           const double* __restrict__ pos, const int32_t* __restrict__ cell_part,
                                           const double* __restrict__ pos_cell, int32_t* keys,
                                           int32_t* __restrict__ list, uint64_t* __restrict__ masks, int nws,
                                           int32_t* __restrict__ counts, int32_t* __restrict__ overflow, int lane) {
    int key[R];
    int sel[6];
#pragma unroll
    for (int b = 0; b < 6; ++b) sel[b] = (lane >> b) & 1 ? INT_MAX : INT_MIN;
#pragma unroll
    for (int r = 0; r < R; ++r) key[r] = lane * R + r < pc.total ? keys[lane * R + r] : INT_MAX;
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
        const bool have = r * kWave + lane < pc.total;
        const int64_t q = have ? key[r] : 0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const float x = relative<DIM>(pc, g, pos[d * n + q], d);
            cx[r][d] = have ? x : 1e18f;  // padding is out of reach
        }
        if (have) list[r * kWave + lane] = key[r];
    }
    const int nw = (pc.total + kWave - 1) >> 6;
    for (int i0 = 0; i0 < pc.np; i0 += kWave) {
        const int m64 = min(kWave, pc.np - i0);
        int pid = 0;
        float xp[DIM];
        if (lane < m64) pid = cell_part[pc.pst + i0 + lane];
#pragma unroll
        for (int d = 0; d < DIM; ++d)
            xp[d] = lane < m64 ? relative<DIM>(pc, g, pos_cell[d * n + pc.pst + i0 + lane], d) : 0.0f;
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
                int nacc = 0;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    float d2 = 0.0f;
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        const float t = cx[r][d] - x[d];
                        d2 = fmaf(t, t, d2);
                    }
                    unsigned long long m = __ballot(d2 < 1.0f + kPairTol) & ~__ballot(key[r] == p);
                    const unsigned long long open = m & __ballot(d2 > 1.0f - kPairTol);
                    if (open) {  // rare: the FP64 formula on the positions themselves
                        double a[3], b[3];
                        const bool mine = (open >> lane) & 1u;
                        const int64_t q = mine ? key[r] : p;
#pragma unroll
                        for (int d = 0; d < DIM; ++d) {
                            a[d] = pos[d * n + p];
                            b[d] = pos[d * n + q];
                        }
                        const bool near = within_cut_at<DIM>(a, b, g, pc.r2);
                        m = (m & ~open) | (open & __ballot(near));
                    }
                    nacc += __popcll(m);
                    wlo = dcpse_writelane((int)m, k * R + r, wlo);
                    whi = dcpse_writelane((int)(m >> 32), k * R + r, whi);
                }
                cnt = dcpse_writelane(nacc, i, cnt);
            }
            if (lane < ie * R && lane % R < nw)
                masks[(pc.pst + i0 + ib + lane / R) * nws + lane % R] = ((uint64_t)(unsigned)whi << 32) | (unsigned)wlo;
        }
        if (lane < m64) {
            counts[pid] = cnt;
            if (cnt > DCPSE_MAX_ROW) atomicOr(overflow, 1);
        }
    }
}

// Count pass: one wavefront per cell (see above); counts[p], the cell's
// sorted candidates at list[c * nws * 64 ..] (ncand[c] of them) and the take
// masks. Cells with more than nws * 64 candidates, and cells with a particle
// far outside (which FP32 would resolve too coarsely), are appended to spill[1 ..] (spill[0] = their number, ncand -1) for
// k_support_cells. RMAX * 64 >= nws * 64 bounds the registers.
//
// Bound by VALU issue: 342 candidates per cell of the 128^3 set with 10%
// removed (rcut 2.4 spacings) shrink to about 170 within reach of the
// particles' bounding box, are sorted in 200-odd instructions, and a pair
// test costs 9 instructions per 64 pairs with the candidates in registers and
// the particle in scalar registers. 0.55 ms there (1.89M particles); FP64
// tests of every candidate from LDS took 1.14 ms, and with them the fill,
// which then sorted every row, 0.96 ms instead of 0.22 ms (k_cell_rows).
template <int DIM, int RMAX>
__global__ __launch_bounds__(kPairWaves * kWave) void k_cell_pairs(
    int64_t n, const double* __restrict__ rcut, CellGrid g, const int64_t* __restrict__ cell_start,
    const int32_t* __restrict__ cell_part, const double* __restrict__ pos_cell, const double* __restrict__ pos,
    int32_t* __restrict__ counts, int32_t* __restrict__ overflow, int32_t* __restrict__ ncand,
    int32_t* __restrict__ lists, uint64_t* __restrict__ masks, int nws, int32_t* __restrict__ spill) {
    __shared__ __align__(16) int32_t kbuf[kPairWaves][RMAX * kWave];
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t c = (int64_t)xcd_block() * kPairWaves + wv;
    if (c >= g.ncell) return;  // whole wavefront
    PairCell<DIM> pc;
    pc.pst = cell_start[c];
    pc.np = (int)(cell_start[c + 1] - pc.pst);
    if (pc.np == 0) return;  // never looked at by the fill either
    int cc[3];
    cell_coords<DIM>(g, c, cc);
    const double r = rcut[0];
    pc.r2 = r * r;
    pc.ir = 1.0 / r;
#pragma unroll
    for (int d = 0; d < DIM; ++d) pc.ctr[d] = g.lo[d] + (cc[d] + 0.5) * g.cs[d];
    // bounding box of the cell's particles
    float lo[DIM], hi[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) lo[d] = 1e30f, hi[d] = 1e30f;  // hi: of the negated coordinate
    const double xmax = kMaxOffset * r;
    bool wild = false;
    for (int i0 = 0; i0 < pc.np; i0 += kWave) {
        const bool have = i0 + lane < pc.np;
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const double xr = have ? pos_cell[d * n + pc.pst + i0 + lane] : 0.0;
            wild |= fabs(xr) > xmax;
            const float x = relative<DIM>(pc, g, xr, d);
            lo[d] = fminf(lo[d], have ? x : 1e30f);
            hi[d] = fminf(hi[d], have ? -x : 1e30f);
        }
    }
    bool spilled = __ballot(wild) != 0;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        lo[d] = wave_min_f(lo[d]);
        hi[d] = -wave_min_f(hi[d]);
        const float far = 2.0f * (float)(g.cs[d] * pc.ir);
        spilled |= !(lo[d] >= -far && hi[d] <= far);
    }
    int nacc = 0;
    if (!spilled) {
        long long cst;
        int ccnt;
        cell_segments<DIM>(g, cell_start, c, lane, cst, ccnt);
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
            int q[4];
            double x[4][DIM];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int k = base + j * kWave + lane;
                const int64_t slot = k < total ? off[j] + k : 0;
                q[j] = cell_part[slot];
#pragma unroll
                for (int d = 0; d < DIM; ++d) x[j][d] = pos_cell[d * n + slot];
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float d2 = 0.0f;  // squared distance to the box
#pragma unroll
                for (int d = 0; d < DIM; ++d) {
                    wild |= fabs(x[j][d]) > xmax;
                    const float a = relative<DIM>(pc, g, x[j][d], d);
                    const float t = fmaxf(fmaxf(lo[d] - a, a - hi[d]), 0.0f);
                    d2 = fmaf(t, t, d2);
                }
                const bool keep = (base + j * kWave + lane < total) & (d2 < 1.0f + 4.0f * kPairTol);
                const unsigned long long m = __ballot(keep);
                const int at = nacc + lane_prefix(m);
                if (keep && at < RMAX * kWave) kbuf[wv][at] = q[j];
                nacc += __popcll(m);
            }
        }
        spilled = nacc > nws * kWave || __ballot(wild) != 0;
    }
    if (spilled) {
        if (lane == 0) {
            spill[1 + atomicAdd(spill, 1)] = (int32_t)c;
            ncand[c] = -1;
        }
        return;
    }
    if (lane == 0) ncand[c] = nacc;
    pc.total = nacc;
    wave_lds_sync();
    int32_t* list = lists + c * nws * kWave;
    if (nacc <= RMAX / 4 * kWave)
        pair_tests<DIM, RMAX / 4>(pc, g, n, pos, cell_part, pos_cell, kbuf[wv], list, masks, nws, counts, overflow,
                                  lane);
    else if (nacc <= RMAX / 2 * kWave)
        pair_tests<DIM, RMAX / 2>(pc, g, n, pos, cell_part, pos_cell, kbuf[wv], list, masks, nws, counts, overflow,
                                  lane);
    else
        pair_tests<DIM, RMAX>(pc, g, n, pos, cell_part, pos_cell, kbuf[wv], list, masks, nws, counts, overflow, lane);
}

// The rows of a cell's particles from its candidate list and the take masks.
template <int R>
__device__ __forceinline__ void pair_rows(int64_t pst, int np, int total, const int32_t* __restrict__ cell_part,
                                          const int32_t* __restrict__ list, const uint64_t* __restrict__ masks, int nws,
                                          int32_t* __restrict__ overflow, const int64_t* __restrict__ row_ptr,
                                          int32_t* __restrict__ col, int lane) {
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
            const int pid = cell_part[pst + i0 + lane];
            rs = row_ptr[pid];
            len = (int)(row_ptr[pid + 1] - rs);
        }
        for (int ib = 0; ib < m64; ib += PER) {
            const int ie = min(PER, m64 - ib);
            uint64_t mw = 0;
            if (lane < ie * R && lane % R < nw) mw = masks[(pst + i0 + ib + lane / R) * nws + lane % R];
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
                    if (lane == 0) atomicOr(overflow, 2);
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

// Fill pass over the cells that k_cell_pairs listed (its cell list, candidate
// lists and masks): a wavefront per cell, four masked stores per row and
// nothing else; bound by the stores and the instructions that address them.
template <int RMAX>
__global__ __launch_bounds__(kPairWaves * kWave) void k_cell_rows(
    int64_t ncell, const int64_t* __restrict__ cell_start, const int32_t* __restrict__ cell_part,
    const int32_t* __restrict__ ncand, const int32_t* __restrict__ lists, const uint64_t* __restrict__ masks, int nws,
    int32_t* __restrict__ overflow, const int64_t* __restrict__ row_ptr, int32_t* __restrict__ col) {
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t c = (int64_t)xcd_block() * kPairWaves + wv;
    if (c >= ncell) return;
    const int64_t pst = cell_start[c];
    const int np = (int)(cell_start[c + 1] - pst);
    if (np == 0) return;
    const int total = ncand[c];
    if (total < 0) return;  // filled from positions
    const int32_t* list = lists + c * nws * kWave;
    if (total <= RMAX / 4 * kWave)
        pair_rows<RMAX / 4>(pst, np, total, cell_part, list, masks, nws, overflow, row_ptr, col, lane);
    else if (total <= RMAX / 2 * kWave)
        pair_rows<RMAX / 2>(pst, np, total, cell_part, list, masks, nws, overflow, row_ptr, col, lane);
    else
        pair_rows<RMAX>(pst, np, total, cell_part, list, masks, nws, overflow, row_ptr, col, lane);
}

// Count (FILL = false: counts[p]) or fill (FILL = true: col[row_ptr[p] ..])
// from positions, one particle of the cell at a time: every cell, or with
// spill != NULL the spill[0] cells listed at spill[1 ..].
template <int DIM, bool FILL>
__global__ __launch_bounds__(kCellWaves * kWave) void k_support_cells(
    int64_t n, const double* __restrict__ rcut, CellGrid g, const int64_t* __restrict__ cell_start,
    const int32_t* __restrict__ cell_part, const double* __restrict__ pos_cell, int32_t* __restrict__ counts,
    int32_t* __restrict__ overflow, const int64_t* __restrict__ row_ptr, int32_t* __restrict__ col,
    const int32_t* __restrict__ spill) {
    constexpr int CAP = CellCap<DIM>::v;
    __shared__ int32_t sq[kCellWaves][CAP];
    __shared__ double sx[kCellWaves][DIM * CAP];
    __shared__ int32_t buf[FILL ? kCellWaves : 1][FILL ? DCPSE_MAX_ROW : 1];
    __shared__ int32_t mark[kCellWaves][kWave];
    __shared__ long long seg_cst[kCellWaves][kWave];
    __shared__ int32_t seg_ex[kCellWaves][kWave];
    const int lane = threadIdx.x & 63;
    const int wv = threadIdx.x >> 6;
    const double r = rcut[0];
    const double r2 = r * r;
    const unsigned G = gridDim.x;
    const int64_t ncells = spill ? (int64_t)spill[0] : g.ncell;
    for (int64_t ci = (int64_t)xcd_block() * kCellWaves + wv; ci < ncells; ci += (int64_t)G * kCellWaves) {
        const int64_t c = spill ? (int64_t)spill[1 + ci] : ci;
        const int64_t pst = cell_start[c];
        const int np = (int)(cell_start[c + 1] - pst);
        if (np == 0) continue;
        long long cst;
        int ccnt;
        cell_segments<DIM>(g, cell_start, c, lane, cst, ccnt);
        const int incl = wave_incl_scan(ccnt);
        const int total = __builtin_amdgcn_readlane(incl, 63);
        const int excl = incl - ccnt;
        seg_cst[wv][lane] = cst;
        seg_ex[wv][lane] = excl;
        const bool fits = total <= CAP;
        if (fits)
            stage_candidates<DIM, true>(0, total, ccnt, excl, mark[wv], seg_cst[wv], seg_ex[wv], cell_part, pos_cell,
                                        n, sq[wv], sx[wv], CAP, lane);
        for (int i = 0; i < np; ++i) {
            const int64_t ps = pst + i;
            const int pid = cell_part[ps];
            double xp[3];
#pragma unroll
            for (int d = 0; d < DIM; ++d) xp[d] = pos_cell[d * n + ps];
            int nacc = 0;
            for (int c0 = 0; c0 < total; c0 += CAP) {
                const int cn = min(CAP, total - c0);
                if (!fits) {
                    wave_lds_sync();
                    stage_candidates<DIM, true>(c0, cn, ccnt, excl, mark[wv], seg_cst[wv], seg_ex[wv], cell_part,
                                                pos_cell, n, sq[wv], sx[wv], CAP, lane);
                }
                for (int t0 = 0; t0 < cn; t0 += kWave) {
                    const int t = min(t0 + lane, cn - 1);
                    const int q = sq[wv][t];
                    const bool near = within_cut<DIM>(xp, sx[wv], CAP, t, g, r2);
                    const bool take = (t0 + lane < cn) & (q != pid) & near;
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
                    counts[pid] = nacc;
                    if (nacc > DCPSE_MAX_ROW) atomicOr(overflow, 1);
                }
            } else {
                wave_lds_sync();
                const int64_t rs = row_ptr[pid];
                const int nn = min(nacc, DCPSE_MAX_ROW);
                if ((int64_t)nacc != row_ptr[pid + 1] - rs) {
                    if (lane == 0) atomicOr(overflow, 2);
                } else {
                    store_ranked(buf[wv], nn, col + rs, lane);
                }
                wave_lds_sync();
            }
        }
        wave_lds_sync();
    }
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

// out[0] = min and out[1] = max(0, max) of v[0..n) (NaNs ignored), one block.
constexpr int kMinMaxThreads = 1024;
__global__ __launch_bounds__(kMinMaxThreads) void k_minmax(const double* __restrict__ v, int64_t n,
                                                          double* __restrict__ out) {
    __shared__ double smin[kMinMaxThreads], smax[kMinMaxThreads];
    const int t = threadIdx.x;
    double lo = n > 0 ? v[0] : 0.0, hi = 0.0;
    for (int64_t i = t; i < n; i += kMinMaxThreads) {
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
        out[0] = smin[0];
        out[1] = smax[0];
    }
}

// Calls launch with the dimension and the register width of a mask of nws
// words as compile-time values.
template <typename F>
static void launch_pairs(int dim, int nws, F launch) {
    auto width = [&](auto D) {
        if (nws <= 4) launch(D, std::integral_constant<int, 4>());
        else if (nws <= 8) launch(D, std::integral_constant<int, 8>());
        else if (nws <= 16) launch(D, std::integral_constant<int, 16>());
        else launch(D, std::integral_constant<int, 32>());
    };
    if (dim == 2) width(std::integral_constant<int, 2>());
    else width(std::integral_constant<int, 3>());
}

static dcpse_status support_pass(dcpse_ctx* ctx, int dim, const double* pos_sup, int64_t n_sup,
                                 const double* pos_dom, int64_t n_dom, const int32_t* dom_self,
                                 const double* rcut, int rcut_pp,
                                 const double* box_lo, const double* box_hi, unsigned periodic,
                                 int64_t* row_ptr, int32_t* col, int64_t* nnz_out) {
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
    // the largest cut-off fixes the cell edge
    double rmax = 0.0, rmin = 0.0;
    if (rcut_pp) {
        // reduced on the device; only the two extremes come back
        Workspace w0;
        dcpse_status st0 = reserve_workspace(ctx, 1024, &w0);
        if (st0) return st0;
        double* mm = w0.take<double>(2);
        k_minmax<<<1, kMinMaxThreads, 0, ctx->stream>>>(rcut, n_dom, mm);
        DCPSE_LAUNCH_CHECK(ctx);
        double h[2] = {0.0, 0.0};
        DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(h, mm, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
        rmin = h[0];
        rmax = h[1];
    } else {
        DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(&rmax, rcut, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(ctx->stream));
        rmin = rmax;
    }
    // cells per cut-off: 2 (3D) or 4 (2D) for one cut-off; with a spread of
    // cut-offs, about rmax / rmin so the smallest scan only their own
    // neighbourhood (bounded: a wave handles 32 cell rows per round)
    const double spread = rmin > 0.0 ? rmax / rmin : 1.0;
    const int K = dim == 3 ? std::min(4, std::max(2, (int)std::ceil(spread - 1e-9)))
                           : std::min(8, std::max(4, (int)std::ceil(spread - 1e-9)));
    CellGrid g;
    dcpse_status st;
    // one particle set and one cut-off: a wavefront per cell of edge >= rcut
    // while the mean candidate count of a cell leaves room to sort them in
    // registers; otherwise a wavefront per particle
    bool by_cell = same && !rcut_pp && n_dom > 0;
    bool paired = false;  // candidate lists and take masks (k_cell_pairs)
    int nws = 0;          // words of a take mask
    if (by_cell) {
        if ((st = make_grid(ctx, dim, box_lo, box_hi, periodic, rmax, 1, &g))) return st;
        const double cand = (double)n_sup * (dim == 3 ? 27.0 : 9.0) / (double)g.ncell;
        by_cell = cand <= (dim == 3 ? 1638.0 : 819.0);
        // about half of the 3^dim cells' particles are within reach of the
        // cell's own; lists of 0.84 of them leave room for uneven cells
        nws = std::max(2, std::min(32, (int)std::ceil(0.84 * cand / kWave)));
        paired = by_cell;
        for (int d = 0; d < dim; ++d) {  // see kPairTol, relative()
            paired = paired && g.cs[d] <= 4.0 * rmax && std::fabs(box_lo[d]) <= kMaxOffset * rmax &&
                     std::fabs(box_hi[d]) <= kMaxOffset * rmax && (g.nc[d] >= 4 || !((periodic >> d) & 1u));
        }
    }
    if (!by_cell && (st = make_grid(ctx, dim, box_lo, box_hi, periodic, rmax, K, &g))) return st;
    const int64_t cb = by_cell ? std::max<int64_t>(1, std::min<int64_t>((g.ncell + kCellWaves - 1) / kCellWaves,
                                                                         (int64_t)ctx->num_cus * 16))
                               : 0;
    const unsigned cell_blocks = (unsigned)(cb >= 8 ? cb / 8 * 8 : cb);
    // one wavefront per cell, the blocks in whole rounds over the XCDs
    const unsigned pair_blocks = (unsigned)((g.ncell + kPairWaves * 8 - 1) / (kPairWaves * 8) * 8);

    // the same-set, single-cut-off fill reuses the cell list, candidate lists and
    // take masks of the count just before it when the arguments match
    dcpse_support_cache& sc = ctx->sup;
    const bool count_pass = col == nullptr;
    const bool cached = paired && !count_pass && sc.valid && sc.dim == dim && sc.pos == pos_sup &&
                        sc.n == n_sup && sc.rcut == rmax && sc.periodic == periodic && sc.nws == nws &&
                        std::equal(box_lo, box_lo + dim, sc.lo) && std::equal(box_hi, box_hi + dim, sc.hi);
    sc.valid = false;

    Workspace w;
    size_t need = (size_t)n_sup * 4 * 2 + (size_t)dim * (n_sup + 1) * 8 + (size_t)(g.ncell + 1) * 8 +
                  (size_t)g.ncell * 4 * 2 + (size_t)n_dom * 4 + scan_workspace_bytes(std::max(g.ncell, n_dom)) +
                  64 * 256;
    if ((st = reserve_workspace(ctx, need, &w))) return st;
    int32_t* cell_id = w.take<int32_t>(n_sup + 1);
    int32_t* cell_part = w.take<int32_t>(n_sup + 1);
    double* pos_cell = w.take<double>((size_t)dim * (n_sup + 1));
    int32_t* cell_cnt = w.take<int32_t>(g.ncell + 1);
    int64_t* cell_start = w.take<int64_t>(g.ncell + 1);
    int32_t* counts = w.take<int32_t>(n_dom + 1);
    int32_t* flags = w.take<int32_t>(64);
    Workspace ws_scan = w;
    if (!flags) return fail(ctx, DCPSE_ERR_INVALID, "workspace sizing error");
    hipStream_t s = ctx->stream;

    uint64_t* masks = nullptr;
    int32_t *spill = nullptr, *ncand = nullptr, *lists = nullptr;
    bool use_cache = paired && (count_pass || cached);
    if (use_cache) {
        // cell list, candidate lists, masks and the list of cells left to the
        // position kernel in the context's support cache
        auto carve = [&](Workspace& cw) {
            cell_start = cw.take<int64_t>(g.ncell + 1);
            cell_part = cw.take<int32_t>(n_sup + 1);
            pos_cell = cw.take<double>((size_t)dim * (n_sup + 1));
            masks = cw.take<uint64_t>((size_t)(n_sup + 1) * nws);
            ncand = cw.take<int32_t>(g.ncell + 1);
            lists = cw.take<int32_t>((size_t)g.ncell * nws * kWave);
            spill = cw.take<int32_t>(g.ncell + 2);
        };
        int64_t* own_start = cell_start;
        int32_t* own_part = cell_part;
        double* own_pos = pos_cell;
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
                use_cache = false;
                cell_start = own_start, cell_part = own_part, pos_cell = own_pos;
                masks = nullptr, spill = nullptr;
            }
        }
        if (use_cache) {
            cw = Workspace();
            cw.base = static_cast<char*>(sc.buf);
            cw.cap = sc.cap;
            carve(cw);
            if (!spill) return fail(ctx, DCPSE_ERR_INVALID, "support cache sizing error");
        }
    }

    fill_i32(s, flags, 64, 0);
    const int64_t tb = std::max<int64_t>(1, std::min<int64_t>((n_sup + 255) / 256, 16384));
    if (!cached) {
        fill_i32(s, cell_cnt, g.ncell + 1, 0);
        if (n_sup > 0) {
            if (dim == 2) k_cell_assign<2><<<(unsigned)tb, 256, 0, s>>>(pos_sup, n_sup, g, cell_id, cell_cnt);
            else k_cell_assign<3><<<(unsigned)tb, 256, 0, s>>>(pos_sup, n_sup, g, cell_id, cell_cnt);
            DCPSE_LAUNCH_CHECK(ctx);
        }
        if ((st = scan_counts(ctx, cell_cnt, g.ncell, cell_start, &ws_scan))) return st;
        fill_i32(s, cell_cnt, g.ncell + 1, 0);  // reuse as cursor
        if (n_sup > 0) {
            if (dim == 2)
                k_cell_fill<2><<<(unsigned)tb, 256, 0, s>>>(cell_id, n_sup, pos_sup, cell_start, cell_cnt,
                                                            cell_part, pos_cell);
            else
                k_cell_fill<3><<<(unsigned)tb, 256, 0, s>>>(cell_id, n_sup, pos_sup, cell_start, cell_cnt,
                                                            cell_part, pos_cell);
            DCPSE_LAUNCH_CHECK(ctx);
        }
    }
    const int64_t rb = std::max<int64_t>(1, std::min<int64_t>((n_dom + kRowWaves - 1) / kRowWaves,
                                                              (int64_t)ctx->num_cus * 16));
    if (count_pass) {
        if (by_cell && !use_cache) {
            if (dim == 2)
                k_support_cells<2, false><<<cell_blocks, kCellWaves * kWave, 0, s>>>(
                    n_sup, rcut, g, cell_start, cell_part, pos_cell, counts, flags, nullptr, nullptr, nullptr);
            else
                k_support_cells<3, false><<<cell_blocks, kCellWaves * kWave, 0, s>>>(
                    n_sup, rcut, g, cell_start, cell_part, pos_cell, counts, flags, nullptr, nullptr, nullptr);
            DCPSE_LAUNCH_CHECK(ctx);
        } else if (by_cell) {
            // candidate lists and masks, then the cells they do not cover from positions
            fill_i32(s, spill, 1, 0);
            launch_pairs(dim, nws, [&](auto D, auto R) {
                k_cell_pairs<decltype(D)::value, decltype(R)::value><<<pair_blocks, kPairWaves * kWave, 0, s>>>(
                    n_sup, rcut, g, cell_start, cell_part, pos_cell, pos_sup, counts, flags, ncand, lists, masks, nws,
                    spill);
            });
            DCPSE_LAUNCH_CHECK(ctx);
            if (dim == 2)
                k_support_cells<2, false><<<cell_blocks, kCellWaves * kWave, 0, s>>>(
                    n_sup, rcut, g, cell_start, cell_part, pos_cell, counts, flags, nullptr, nullptr, spill);
            else
                k_support_cells<3, false><<<cell_blocks, kCellWaves * kWave, 0, s>>>(
                    n_sup, rcut, g, cell_start, cell_part, pos_cell, counts, flags, nullptr, nullptr, spill);
            DCPSE_LAUNCH_CHECK(ctx);
        } else if (n_dom > 0) {
            if (dim == 2)
                k_support_rows<2, false><<<(unsigned)rb, kRowWaves * kWave, 0, s>>>(
                    pos_sup, n_sup, pos_dom, n_dom, same, dom_self, rcut, rcut_pp, g, cell_start, cell_part, pos_cell, counts,
                    flags, nullptr, nullptr);
            else
                k_support_rows<3, false><<<(unsigned)rb, kRowWaves * kWave, 0, s>>>(
                    pos_sup, n_sup, pos_dom, n_dom, same, dom_self, rcut, rcut_pp, g, cell_start, cell_part, pos_cell, counts,
                    flags, nullptr, nullptr);
            DCPSE_LAUNCH_CHECK(ctx);
        }
        Workspace ws2 = ws_scan;
        if ((st = scan_counts(ctx, counts, n_dom, row_ptr, &ws2))) return st;
        int64_t nnz = 0;
        int32_t ovf = 0, n_spill = 0;
        DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(&nnz, row_ptr + n_dom, sizeof(int64_t), hipMemcpyDeviceToHost, s));
        DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(&ovf, flags, sizeof(int32_t), hipMemcpyDeviceToHost, s));
        if (spill)
            DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(&n_spill, spill, sizeof(int32_t), hipMemcpyDeviceToHost, s));
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(s));
        if (ovf & 1)
            return fail(ctx, DCPSE_ERR_RANGE, "a support row exceeds DCPSE_MAX_ROW=%d neighbours",
                        DCPSE_MAX_ROW);
        if (nnz >= ((int64_t)1 << 31) * 64)
            return fail(ctx, DCPSE_ERR_RANGE, "nnz out of range");
        if (nnz_out) *nnz_out = nnz;
        if (use_cache) {
            sc.valid = true;
            sc.spill = n_spill > 0;
            sc.dim = dim;
            sc.pos = pos_sup;
            sc.n = n_sup;
            sc.rcut = rmax;
            sc.periodic = periodic;
            sc.nws = nws;
            for (int d = 0; d < 3; ++d) {
                sc.lo[d] = d < dim ? box_lo[d] : 0.0;
                sc.hi[d] = d < dim ? box_hi[d] : 0.0;
            }
        }
    } else {
        if (cached) {
            launch_pairs(dim, nws, [&](auto, auto R) {
                k_cell_rows<decltype(R)::value><<<pair_blocks, kPairWaves * kWave, 0, s>>>(
                    g.ncell, cell_start, cell_part, ncand, lists, masks, nws, flags, row_ptr, col);
            });
            DCPSE_LAUNCH_CHECK(ctx);
        }
        if (by_cell && (!cached || sc.spill)) {
            // the cells the lists do not cover (cached), or all of them
            const int32_t* list = cached ? spill : nullptr;
            if (dim == 2)
                k_support_cells<2, true><<<cell_blocks, kCellWaves * kWave, 0, s>>>(
                    n_sup, rcut, g, cell_start, cell_part, pos_cell, counts, flags, row_ptr, col, list);
            else
                k_support_cells<3, true><<<cell_blocks, kCellWaves * kWave, 0, s>>>(
                    n_sup, rcut, g, cell_start, cell_part, pos_cell, counts, flags, row_ptr, col, list);
            DCPSE_LAUNCH_CHECK(ctx);
        } else if (!by_cell && n_dom > 0) {
            if (dim == 2)
                k_support_rows<2, true><<<(unsigned)rb, kRowWaves * kWave, 0, s>>>(
                    pos_sup, n_sup, pos_dom, n_dom, same, dom_self, rcut, rcut_pp, g, cell_start, cell_part, pos_cell, counts,
                    flags, row_ptr, col);
            else
                k_support_rows<3, true><<<(unsigned)rb, kRowWaves * kWave, 0, s>>>(
                    pos_sup, n_sup, pos_dom, n_dom, same, dom_self, rcut, rcut_pp, g, cell_start, cell_part, pos_cell, counts,
                    flags, row_ptr, col);
            DCPSE_LAUNCH_CHECK(ctx);
        }
        if (n_dom > 0) {
            const int64_t lb = std::max<int64_t>(
                1, std::min<int64_t>((n_dom + kRowWaves * kWave - 1) / (kRowWaves * kWave), (int64_t)ctx->num_cus * 8));
            k_sort_long_rows<<<(unsigned)lb, kRowWaves * kWave, 0, s>>>(n_dom, row_ptr, col);
            DCPSE_LAUNCH_CHECK(ctx);
        }
        int32_t ovf = 0;
        DCPSE_HIP_CHECK(ctx, hipMemcpyAsync(&ovf, flags, sizeof(int32_t), hipMemcpyDeviceToHost, s));
        DCPSE_HIP_CHECK(ctx, hipStreamSynchronize(s));
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
