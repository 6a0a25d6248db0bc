// DC-PSE operator application for gfx950: CSR neighbour gather.
//
// Restates the bulk apply of src/DCPSE/Dcpse.hpp:467-499 (and the per-key
// form :560-659 that the expression nodes of
// src/DCPSE/DCPSE_op/DCPSE_op.hpp:64-67 and :389-401 call) as
//     Df_p = sum_q W_pq (f_q - f_p),   W = eps_p^-|beta| K_pq (pre-scaled),
// the difference form: for odd |beta| the constant monomial is in the basis
// and its moment condition gives sum_q K_pq = 0, so the reference's
// (f_q + f_p) equals (f_q - f_p) up to rounding; for even |beta| it is the
// reference's own sign.
//
// The kernel is HBM-bound (about 8 bytes per nonzero per operator). G lanes
// cooperate on one row so the W/col streams are read as contiguous segments;
// several operators sharing one support (e.g. Laplacian and Dx) and several
// fields share the col stream and the f gather in one pass. Workgroups are
// remapped so that each XCD walks one contiguous slice of rows, keeping the
// f halo of a slice in that XCD's L2.
#include <algorithm>
#include <cstdint>
#include <optional>
#include <type_traits>

#include "dcpse_common.hpp"
#include "dcpse_internal.hpp"

namespace dcpse {

// Loads of the col/W streams: ordinary cached loads (rows are not aligned to
// cache lines, so a line split between two load instructions is found in L2 by
// the second).
#define DCPSE_STREAM_LOAD(p) (*(p))

constexpr int kMaxOps = 4;

template <typename T>
struct ApplyArgs {
    int64_t n_rows;
    const int64_t* row_ptr;
    const int32_t* col;
    const T* W[kMaxOps];
    const T* f;
    int64_t ld_f;
    const T* f_self;
    int64_t ld_self;
    const T* diag;  // transpose mode only
    T* out[kMaxOps];
    int64_t ld_out;
    T alpha, beta;
    int64_t blocks_needed;  // logical blocks
    int64_t per_xcd;        // logical blocks per XCD slice
};

enum ApplyMode { kDiff = 0, kExplicitDiag = 1 };

constexpr int kApplyMaxBlock = 512;  // launch bound of k_apply; larger blocks are rejected

// G lanes cooperate on one row. The first G*EPL nonzeros of the row are
// handled with every load issued before any is consumed: EPL col and
// NOPS*EPL weight loads per lane (indices clamped into the row, so no branch
// separates them), then EPL gathers of f, then the FMAs. Longer rows finish
// in a strided loop. Invalid (clamped) slots are masked out by a select.
template <typename T, int G, int EPL, int NOPS, int NF, int MODE>
__global__ __launch_bounds__(kApplyMaxBlock) void k_apply(const ApplyArgs<T> a) {
    // XCD-aware remap: hardware block b runs on XCD b % 8; give each XCD a
    // contiguous range of logical blocks.
    const int64_t hb = blockIdx.x;
    const int64_t lb = (hb & 7) * a.per_xcd + (hb >> 3);
    if (lb >= a.blocks_needed) return;
    const int rows_per_block = blockDim.x / G;
    const int gl = threadIdx.x % G;
    const int64_t row = lb * rows_per_block + threadIdx.x / G;
    if (row >= a.n_rows) return;  // whole G-lane groups leave together
    const int64_t rs = a.row_ptr[row];
    const int64_t re = a.row_ptr[row + 1];
    T fp[NF];
#pragma unroll
    for (int b = 0; b < NF; ++b) fp[b] = a.f_self[b * a.ld_self + row];
    double acc[NOPS][NF];  // FP64 accumulation for both value types
#pragma unroll
    for (int o = 0; o < NOPS; ++o)
#pragma unroll
        for (int b = 0; b < NF; ++b) acc[o][b] = 0.0;
    if (re > rs) {
        int32_t q[EPL];
        T w[NOPS][EPL];
        bool v[EPL];
#pragma unroll
        for (int k = 0; k < EPL; ++k) {
            const int64_t j = rs + gl + k * G;
            v[k] = j < re;
            const int64_t jj = v[k] ? j : re - 1;
            q[k] = DCPSE_STREAM_LOAD(a.col + jj);
#pragma unroll
            for (int o = 0; o < NOPS; ++o) w[o][k] = DCPSE_STREAM_LOAD(a.W[o] + jj);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < NF; ++b) {
            T fq[EPL];
#pragma unroll
            for (int k = 0; k < EPL; ++k) fq[k] = a.f[b * a.ld_f + q[k]];
#pragma unroll
            for (int k = 0; k < EPL; ++k) {
                const double d = MODE == kDiff ? (double)fq[k] - (double)fp[b] : (double)fq[k];
#pragma unroll
                for (int o = 0; o < NOPS; ++o) acc[o][b] = v[k] ? fma((double)w[o][k], d, acc[o][b]) : acc[o][b];
            }
        }
        for (int64_t j = rs + gl + G * EPL; j < re; j += G) {
            const int32_t qq = DCPSE_STREAM_LOAD(a.col + j);
            T ww[NOPS];
#pragma unroll
            for (int o = 0; o < NOPS; ++o) ww[o] = DCPSE_STREAM_LOAD(a.W[o] + j);
#pragma unroll
            for (int b = 0; b < NF; ++b) {
                const T fq = a.f[b * a.ld_f + qq];
                const double d = MODE == kDiff ? (double)fq - (double)fp[b] : (double)fq;
#pragma unroll
                for (int o = 0; o < NOPS; ++o) acc[o][b] = fma((double)ww[o], d, acc[o][b]);
            }
        }
    }
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1)
#pragma unroll
        for (int o = 0; o < NOPS; ++o)
#pragma unroll
            for (int b = 0; b < NF; ++b) acc[o][b] += __shfl_xor(acc[o][b], off, kWave);
    if (gl == 0) {
#pragma unroll
        for (int o = 0; o < NOPS; ++o)
#pragma unroll
            for (int b = 0; b < NF; ++b) {
                double val = acc[o][b];
                if (MODE == kExplicitDiag) val = fma((double)a.diag[row], (double)fp[b], val);
                T* dst = a.out[o] + b * a.ld_out + row;
                val *= (double)a.alpha;
                if (a.beta != T(0)) val = fma((double)a.beta, (double)*dst, val);
                *dst = (T)val;
            }
    }
}

// 4-byte-aligned 4-vectors: one 16-byte load per lane at any element offset.
typedef int32_t vi4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float vf4u __attribute__((ext_vector_type(4), aligned(4)));

// FP32 variant: each lane loads 4 consecutive nonzeros of its row with one
// 16-byte load per stream (col and every weight array), so a wavefront
// instruction moves a contiguous 64*G-byte segment per row. NCH such chunks per
// lane are issued before the gathers; longer rows finish in a strided loop.
// The last rows of the CSR, whose 16-byte loads could pass the end of the
// arrays, take the scalar path.
template <int G, int NCH, int NOPS, int NF, int MODE>
__global__ __launch_bounds__(kApplyMaxBlock) void k_apply_v4(const ApplyArgs<float> a) {
    const int64_t hb = blockIdx.x;
    const int64_t lb = (hb & 7) * a.per_xcd + (hb >> 3);
    if (lb >= a.blocks_needed) return;
    const int rows_per_block = blockDim.x / G;
    const int gl = threadIdx.x % G;
    const int64_t row = lb * rows_per_block + threadIdx.x / G;
    if (row >= a.n_rows) return;
    const int64_t rs = a.row_ptr[row];
    const int64_t re = a.row_ptr[row + 1];
    const int64_t nnz_total = a.row_ptr[a.n_rows];
    float fp[NF];
#pragma unroll
    for (int b = 0; b < NF; ++b) fp[b] = a.f_self[b * a.ld_self + row];
    double acc[NOPS][NF];  // FP64 accumulation of the FP32 products
#pragma unroll
    for (int o = 0; o < NOPS; ++o)
#pragma unroll
        for (int b = 0; b < NF; ++b) acc[o][b] = 0.0;
    int64_t jtail = rs + gl;  // first element of the strided scalar loop
    // 16-byte loads read elements e..e+3 with e <= re-1, so re + 3 <= nnz_total
    // keeps them inside the arrays; empty rows skip the vector section.
    if (re > rs && re + 3 <= nnz_total) {
        vi4u q[NCH];
        vf4u w[NOPS][NCH];
        int64_t e0[NCH];
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            e0[c] = rs + 4 * (gl + c * G);
            const int64_t ee = e0[c] < re ? e0[c] : re - 1;  // clamped chunks are masked below
            q[c] = DCPSE_STREAM_LOAD((const vi4u*)(a.col + ee));
#pragma unroll
            for (int o = 0; o < NOPS; ++o) w[o][c] = DCPSE_STREAM_LOAD((const vf4u*)(a.W[o] + ee));
        }
        // keep every stream load ahead of the gathers that depend on col
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < NF; ++b) {
            float fq[NCH][4];
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                fq[c][0] = a.f[b * a.ld_f + q[c].x];
                fq[c][1] = a.f[b * a.ld_f + q[c].y];
                fq[c][2] = a.f[b * a.ld_f + q[c].z];
                fq[c][3] = a.f[b * a.ld_f + q[c].w];
            }
#pragma unroll
            for (int c = 0; c < NCH; ++c)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool v = e0[c] + i < re;
                    const double d = MODE == kDiff ? (double)fq[c][i] - (double)fp[b] : (double)fq[c][i];
#pragma unroll
                    for (int o = 0; o < NOPS; ++o) acc[o][b] = v ? fma((double)w[o][c][i], d, acc[o][b]) : acc[o][b];
                }
        }
        jtail = rs + 4 * G * NCH + gl;
    }
    for (int64_t j = jtail; j < re; j += G) {
        const int32_t qq = DCPSE_STREAM_LOAD(a.col + j);
        float ww[NOPS];
#pragma unroll
        for (int o = 0; o < NOPS; ++o) ww[o] = DCPSE_STREAM_LOAD(a.W[o] + j);
#pragma unroll
        for (int b = 0; b < NF; ++b) {
            const float fq = a.f[b * a.ld_f + qq];
            const double d = MODE == kDiff ? (double)fq - (double)fp[b] : (double)fq;
#pragma unroll
            for (int o = 0; o < NOPS; ++o) acc[o][b] = fma((double)ww[o], d, acc[o][b]);
        }
    }
#pragma unroll
    for (int off = G / 2; off > 0; off >>= 1)
#pragma unroll
        for (int o = 0; o < NOPS; ++o)
#pragma unroll
            for (int b = 0; b < NF; ++b) acc[o][b] += __shfl_xor(acc[o][b], off, kWave);
    if (gl == 0) {
#pragma unroll
        for (int o = 0; o < NOPS; ++o)
#pragma unroll
            for (int b = 0; b < NF; ++b) {
                double val = acc[o][b];
                if (MODE == kExplicitDiag) val = fma((double)a.diag[row], (double)fp[b], val);
                float* dst = a.out[o] + b * a.ld_out + row;
                val *= (double)a.alpha;
                if (a.beta != 0.0f) val = fma((double)a.beta, (double)*dst, val);
                *dst = (float)val;
            }
    }
}

// Batches of FP32 fields on one set: the NF fields are first interleaved
// particle-major (fil[q * NF + b]), so a neighbour's NF values are one
// contiguous 4 NF-byte read instead of NF separate gathers, and the col/W
// streams are read once for all of them; nf <= NF fields, zeros for the rest.
// Each field's sum runs over the nonzeros in the order of k_apply_v4, so the
// results equal the field-major kernel's bit for bit.
template <int NF, typename T>
__global__ __launch_bounds__(256) void k_interleave(int64_t n, const T* __restrict__ f, int64_t ld, int nf,
                                                    T* __restrict__ fil) {
    __shared__ T t[NF][257];
    const int64_t q0 = (int64_t)blockIdx.x * 256;
    const int64_t q = q0 + threadIdx.x;
#pragma unroll
    for (int b = 0; b < NF; ++b) t[b][threadIdx.x] = q < n && b < nf ? f[b * ld + q] : T(0);
    __syncthreads();
    for (int k = threadIdx.x; k < 256 * NF; k += 256) {
        const int qq = k / NF, b = k % NF;
        if (q0 + qq < n) fil[(q0 + qq) * NF + b] = t[b][qq];
    }
}

typedef float vf4a __attribute__((ext_vector_type(4)));

// EL consecutive 4-byte elements of a stream, at any element offset.
template <typename T, int EL>
struct StreamVec {
    typedef T type __attribute__((ext_vector_type(EL), aligned(4)));
};
template <typename T>
struct StreamVec<T, 1> {
    typedef T type;
};

// v of lane SRC of this lane's group of L lanes (L = 1, 2, 4).
template <int L, int SRC>
__device__ __forceinline__ int group_lane(int v) {
    if constexpr (L == 1) return v;
    else if constexpr (L == 2) return __builtin_amdgcn_update_dpp(0, v, SRC ? 0xF5 : 0xA0, 0xF, 0xF, true);
    else return __builtin_amdgcn_update_dpp(0, v, SRC * 0x55, 0xF, 0xF, true);
}

// R = 4 or 8 lanes per row: L = NF / 4 of them side by side hold 4 fields each,
// so one 16-byte load instruction serves 64 / L neighbours with one cache line
// each, and H = R / L such parts share the row's partial sums. (With a lane per
// neighbour reading all its NF values, every one of its 16-byte loads looked up
// 64 lines: 308 us against 161 us forward, 395 against 175 us transposed, for
// 16 fields on 1024^2 particles with 29 neighbours. The cache's lookup rate
// bounded that; here the vector units and the address unit are busy two thirds
// of the time each. Measured and not better: more waves (spilled registers),
// the next chunk's gathers ahead of the sums (half the waves), 32-bit
// addresses; and for 4 and 8 fields one part of 1 and 2 lanes per row, whose
// partial sums follow one another: 100 us against the 56 us of a lane per
// neighbour for 6 fields on 512^2 particles.) A part's lanes load a chunk of 4
// nonzeros together and pass them round by DPP. Each field's sum takes the
// order of k_apply_v4<G, NCH>, whose lane p of a row sums the chunks p, p + G,
// ... and then the strided tail: part h forms the partial sums h, h + H, ...
// one after another, and all are added up as that kernel's lane exchanges do,
// the last exchanges between the parts.
template <int G, int NCH, int NF, int MODE, int R>
struct BatchRow {
    static constexpr int L = NF / 4, EL = 4 / L, H = R / L, GP = G / H;
    static_assert(H <= G, "a part has at least one partial sum");
    typedef typename StreamVec<int32_t, EL>::type vq;
    typedef typename StreamVec<float, EL>::type vw;
    const ApplyArgs<float>& a;
    int64_t rs;
    int len, lenv;  // nonzeros; those taken in chunks of 4 (0: all by the tail)
    int g, h;       // lane of its part, part
    vf4a fp;
    // the chunks' columns and weights, read ahead while they fit 48 registers
    static constexpr bool AHEAD = 2 * EL * GP * NCH <= 48;
    vq q[AHEAD ? GP * NCH : 1];
    vw w[AHEAD ? GP * NCH : 1];

    template <int K>
    __device__ __forceinline__ void element(int32_t qv, float wv, vf4a& f, double& wd) {
        const int32_t qq = group_lane<L, K>(qv);
        wd = (double)__int_as_float(group_lane<L, K>(__float_as_int(wv)));
        f = *reinterpret_cast<const vf4a*>(a.f + ((int64_t)qq * NF + 4 * g));
    }
    static __device__ __forceinline__ int32_t part(const vq& v, int k) {
        if constexpr (EL == 1) return v;
        else return v[k];
    }
    static __device__ __forceinline__ float part(const vw& v, int k) {
        if constexpr (EL == 1) return v;
        else return v[k];
    }
    template <bool MASK>
    __device__ __forceinline__ void add(const vf4a (&f)[4], const double (&wd)[4], const bool (&v)[4], double (&s)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const double d = MODE == kDiff ? (double)f[i][b] - (double)fp[b] : (double)f[i][b];
                const double t = fma(wd[i], d, s[b]);
                s[b] = MASK ? (v[i] ? t : s[b]) : t;
            }
    }
    template <bool MASK>
    __device__ __forceinline__ void four(const vq& qc, const vw& wc, const bool (&v)[4], double (&s)[4]) {
        vf4a f[4];
        double wd[4];
        element<0 / EL>(part(qc, 0 % EL), part(wc, 0 % EL), f[0], wd[0]);
        element<1 / EL>(part(qc, 1 % EL), part(wc, 1 % EL), f[1], wd[1]);
        element<2 / EL>(part(qc, 2 % EL), part(wc, 2 % EL), f[2], wd[2]);
        element<3 / EL>(part(qc, 3 % EL), part(wc, 3 % EL), f[3], wd[3]);
        add<MASK>(f, wd, v, s);
    }
    // First nonzero of the part's C-th chunk.
    template <int C>
    __device__ __forceinline__ int first() const {
        return H == 1 ? 4 * C : 4 * (C * H + h);
    }
    // Column and weight of that chunk: lane g takes EL of its 4 nonzeros.
    template <int C>
    __device__ __forceinline__ void load(vq& qc, vw& wc) {
        const int e = first<C>() + EL * g;
        const int64_t at = lenv > 0 ? rs + min(e, lenv - 1) : 0;
        qc = *reinterpret_cast<const vq*>(a.col + at);
        wc = *reinterpret_cast<const vw*>(a.W[0] + at);
    }
    template <int C>
    __device__ __forceinline__ void load_ahead() {
        if constexpr (AHEAD) {
            if (__ballot(first<C>() < lenv)) load<C>(q[C], w[C]);
            if constexpr (C + 1 < GP * NCH) load_ahead<C + 1>();
        }
    }
    template <int C>
    __device__ __forceinline__ void chunk(double (&s)[4]) {
        const int e = first<C>();
        if (!__ballot(e < lenv)) return;
        const bool v[4] = {e < lenv, e + 1 < lenv, e + 2 < lenv, e + 3 < lenv};
        vq qc;
        vw wc;
        if constexpr (AHEAD) qc = q[C], wc = w[C];
        else load<C>(qc, wc);
        if (__ballot(!v[3])) four<true>(qc, wc, v, s);
        else four<false>(qc, wc, v, s);
    }
    // EL of the four nonzeros e, e + G, ... of the tail.
    __device__ __forceinline__ void load_tail(int e, vq& qv, vw& wv) {
        int32_t qe[EL];
        float we[EL];
#pragma unroll
        for (int k = 0; k < EL; ++k) {
            const int at = e + G * (EL * g + k);
            const int64_t j = at < len ? rs + at : 0;
            qe[k] = a.col[j];
            we[k] = a.W[0][j];
        }
        if constexpr (EL == 1) qv = qe[0], wv = we[0];
        else
#pragma unroll
            for (int k = 0; k < EL; ++k) qv[k] = qe[k], wv[k] = we[k];
    }
    // The part's P-th partial sum: its chunks, then every G-th nonzero of the
    // tail, whose columns and weights are read one step ahead.
    template <int P>
    __device__ __forceinline__ void partial(double (&s)[4]) {
#pragma unroll
        for (int b = 0; b < 4; ++b) s[b] = 0.0;
        int e = (lenv > 0 ? 4 * G * NCH : 0) + (H == 1 ? P : P * H + h);
        vq qt, qn;
        vw wt, wn;
        bool more = __ballot(e < len) != 0;
        if (more) load_tail(e, qt, wt);
        chunk<P>(s);
        if constexpr (NCH > 1) chunk<P + GP>(s);
        if constexpr (NCH > 2) chunk<P + 2 * GP>(s);
        while (more) {
            more = __ballot(e + 4 * G < len) != 0;
            if (more) load_tail(e + 4 * G, qn, wn);
            const bool v[4] = {e < len, e + G < len, e + 2 * G < len, e + 3 * G < len};
            four<true>(qt, wt, v, s);
            e += 4 * G;
            qt = qn;
            wt = wn;
        }
    }
    // The sum that lane P * H + h of k_apply_v4's row holds after exchanges at
    // distances G/2 .. OFF * H.
    template <int P, int OFF>
    __device__ __forceinline__ void tree(double (&s)[4]) {
        if constexpr (OFF == GP) {
            partial<P>(s);
        } else {
            tree<P, 2 * OFF>(s);
            double t[4];
            tree<P + OFF, 2 * OFF>(t);
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                s[b] += t[b];
                asm volatile("" : "+v"(s[b]));  // added here: not all partial sums kept to the end
            }
        }
    }
};

constexpr int kBatchBlock = 256;
constexpr int kBatchMin = 3;  // fields that go particle-major
template <int G, int NCH, int NF, int MODE, int R>
__global__ __launch_bounds__(kBatchBlock) void k_apply_batch(const ApplyArgs<float> a, int nf) {
    typedef BatchRow<G, NCH, NF, MODE, R> Row;
    const int64_t hb = blockIdx.x;
    const int64_t lb = (hb & 7) * a.per_xcd + (hb >> 3);
    if (lb >= a.blocks_needed) return;
    const int64_t at = (lb * kBatchBlock + threadIdx.x) / R;
    const bool live = at < a.n_rows;
    if (!__ballot(live)) return;  // whole wavefront
    const int64_t row = live ? at : a.n_rows - 1;
    const int64_t nnz_total = a.row_ptr[a.n_rows];
    const int64_t re = a.row_ptr[row + 1];
    Row r{a};
    r.rs = a.row_ptr[row];
    r.len = (int)(re - r.rs);
    // rows whose vector loads could pass the end of the arrays take the tail's
    // single loads, as in k_apply_v4
    r.lenv = re + 3 <= nnz_total ? r.len : 0;
    r.g = threadIdx.x % Row::L;
    r.h = threadIdx.x % R / Row::L;
    r.fp = *reinterpret_cast<const vf4a*>(a.f + row * NF + 4 * r.g);
    double s[4];
    r.template load_ahead<0>();
    r.template tree<0, 1>(s);
    // the parts' sums: lane ^ 4, ^ 2, ^ 1 of the row's
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        if constexpr (R == 8) s[b] += __shfl_xor(s[b], 4, kWave);
        if constexpr (Row::L <= 2 && R >= 4) s[b] += dpp_d<0x4E>(s[b]);
        if constexpr (Row::L == 1) s[b] += dpp_d<0xB1>(s[b]);
    }
    if (!live) return;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        if (r.h != (Row::H <= 4 ? b * Row::H / 4 : b) || 4 * r.g + b >= nf) continue;  // another part's, or none
        double val = s[b];
        if (MODE == kExplicitDiag) val = fma((double)a.diag[row], (double)r.fp[b], val);
        float* dst = a.out[0] + (4 * r.g + b) * a.ld_out + row;
        val *= (double)a.alpha;
        if (a.beta != 0.0f) val = fma((double)a.beta, (double)*dst, val);
        *dst = (float)val;
    }
}

template <int G, int NCH, int NF, int MODE, int R>
static void launch_batch(ApplyArgs<float> a, int nf, hipStream_t s) {
    const int rows_per_block = kBatchBlock / R;
    a.blocks_needed = (a.n_rows + rows_per_block - 1) / rows_per_block;
    a.per_xcd = (a.blocks_needed + 7) / 8;
    k_apply_batch<G, NCH, NF, MODE, R><<<(unsigned)(a.per_xcd * 8), kBatchBlock, 0, s>>>(a, nf);
}

// Eight lanes per row where rows are long or few, four otherwise (us, 4 / 8
// lanes; B16: 16 fields, B4: 4). Few rows leave waves to spare: 91,000 rows of
// 62 B16 48 / 41, of 93 65 / 53; 131,000 of 29 35 / 33. Long ones: 729,000 of 93
// B16 438 / 342, B4 195 / 173; 512,000 of 62 202 / 171, 85 / 84; 490,000 of 51
// 142 / 127 but B4 54 / 57; 1,049,000 of 29 187 / 198, 89 / 106.
template <int G, int NCH, int NF, int MODE>
static void launch_apply_il(const ApplyArgs<float>& a, int nf, double mean, hipStream_t s) {
    if constexpr (G == 8) {
        if (a.n_rows <= 131072 || mean > (NF == 16 ? 40.0 : 56.0))
            return launch_batch<G, NCH, NF, MODE, 8>(a, nf, s);
    }
    launch_batch<G, NCH, NF, MODE, 4>(a, nf, s);
}

// FP64 batches: eight lanes per row, NF / 2 of them side by side with two
// fields each (one 16-byte load per lane, a neighbour's NF values in one line),
// the row's nonzeros dealt to the H = 16 / NF parts. Nonzero j belongs to
// partial sum j % G, as in k_apply<double, G, EPL> whose lanes' exchanges add
// them up: part h holds the sums h, h + H, ..., so every field equals the
// single-field CSR kernel bit for bit. (us per apply, 4 fields at a time
// field-major / so: 262,000 rows of 29 B4 53 / 33, B16 207 / 92; 729,000 of 93
// B4 321 / 319, B16 1287 / 920.)
template <int NF, int G, int MODE>
__global__ __launch_bounds__(kBatchBlock) void k_apply_batch64(const ApplyArgs<double> a, int nf) {
    constexpr int L = NF / 2, H = 8 / L, S = G / H, U = S < 4 ? 4 : S < 8 ? S : 8;
    static_assert(S % U == 0 || U % S == 0, "a step takes whole turns of the partial sums");
    constexpr int STEP = S > U ? S : U;  // of the part's nonzeros
    const int64_t hb = blockIdx.x;
    const int64_t lb = (hb & 7) * a.per_xcd + (hb >> 3);
    if (lb >= a.blocks_needed) return;
    const int64_t at = (lb * kBatchBlock + threadIdx.x) / 8;
    const bool live = at < a.n_rows;
    const int64_t row = live ? at : a.n_rows - 1;
    const int g = threadIdx.x % L, h = threadIdx.x % 8 / L;
    const int64_t rs = a.row_ptr[row];
    const int len = live ? (int)(a.row_ptr[row + 1] - rs) : 0;
    const double2 fp = *reinterpret_cast<const double2*>(a.f + row * NF + 2 * g);
    double sx[S], sy[S];
#pragma unroll
    for (int i = 0; i < S; ++i) sx[i] = sy[i] = 0.0;
    for (int j0 = h; j0 < len; j0 += H * STEP) {
#pragma unroll
        for (int k0 = 0; k0 < STEP; k0 += U) {
            int32_t q[U];
            double w[U];
            double2 f[U];
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const int64_t j = rs + min(j0 + H * (k0 + k), len - 1);
                q[k] = a.col[j];
                w[k] = a.W[0][j];
            }
#pragma unroll
            for (int k = 0; k < U; ++k) f[k] = *reinterpret_cast<const double2*>(a.f + (int64_t)q[k] * NF + 2 * g);
#pragma unroll
            for (int k = 0; k < U; ++k) {
                const bool in = j0 + H * (k0 + k) < len;
                const int i = (k0 + k) % S;
                const double tx = fma(w[k], MODE == kDiff ? f[k].x - fp.x : f[k].x, sx[i]);
                const double ty = fma(w[k], MODE == kDiff ? f[k].y - fp.y : f[k].y, sy[i]);
                sx[i] = in ? tx : sx[i];
                sy[i] = in ? ty : sy[i];
            }
        }
    }
    // distances G/2 .. H inside the part, H/2 .. 1 between the parts
#pragma unroll
    for (int off = S / 2; off > 0; off >>= 1)
#pragma unroll
        for (int i = 0; i < off; ++i) {
            sx[i] += sx[i + off];
            sy[i] += sy[i + off];
        }
#pragma unroll
    for (int off = 4; off >= L; off >>= 1) {
        sx[0] += __shfl_xor(sx[0], off, kWave);
        sy[0] += __shfl_xor(sy[0], off, kWave);
    }
    if (!live || h >= 2) return;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        if ((H > 1 && b != h % 2) || 2 * g + b >= nf) continue;  // the other part's field, or none
        double val = b ? sy[0] : sx[0];
        if (MODE == kExplicitDiag) val = fma(a.diag[row], b ? fp.y : fp.x, val);
        double* dst = a.out[0] + (2 * g + b) * a.ld_out + row;
        val *= a.alpha;
        if (a.beta != 0.0) val = fma(a.beta, *dst, val);
        *dst = val;
    }
}

template <int NF, int MODE>
static void launch_batch64(ApplyArgs<double> a, int nf, int G, hipStream_t s) {
    const int rows_per_block = kBatchBlock / 8;
    a.blocks_needed = (a.n_rows + rows_per_block - 1) / rows_per_block;
    a.per_xcd = (a.blocks_needed + 7) / 8;
    const unsigned grid = (unsigned)(a.per_xcd * 8);
    if (G == 16) k_apply_batch64<NF, 16, MODE><<<grid, kBatchBlock, 0, s>>>(a, nf);
    else k_apply_batch64<NF, 8, MODE><<<grid, kBatchBlock, 0, s>>>(a, nf);
}

// The interleaved batch kernel for the shapes of the 16-byte-load kernel
// (il_shape: whether one exists).
static bool il_shape(int G, int epl) {
    return (G == 4 && epl == 8) || (G == 8 && (epl == 4 || epl == 8 || epl == 12)) ||
           (G == 16 && (epl == 4 || epl == 8)) || (G == 32 && epl == 4);
}
template <int MODE, int NF>
static bool dispatch_il(const ApplyArgs<float>& a, int G, int epl, int nf, double mean, hipStream_t s) {
    if (G == 4 && epl == 8) return launch_apply_il<4, 2, NF, MODE>(a, nf, mean, s), true;
    if (G == 8 && epl == 4) return launch_apply_il<8, 1, NF, MODE>(a, nf, mean, s), true;
    if (G == 8 && epl == 8) return launch_apply_il<8, 2, NF, MODE>(a, nf, mean, s), true;
    if (G == 8 && epl == 12) return launch_apply_il<8, 3, NF, MODE>(a, nf, mean, s), true;
    if (G == 16 && epl == 4) return launch_apply_il<16, 1, NF, MODE>(a, nf, mean, s), true;
    if (G == 16 && epl == 8) return launch_apply_il<16, 2, NF, MODE>(a, nf, mean, s), true;
    if (G == 32 && epl == 4) return launch_apply_il<32, 1, NF, MODE>(a, nf, mean, s), true;
    return false;
}

template <typename T, int G, int EPL, int NOPS, int NF, int MODE>
static void launch_apply(ApplyArgs<T> a, int block, hipStream_t s) {
    const int rows_per_block = block / G;
    a.blocks_needed = (a.n_rows + rows_per_block - 1) / rows_per_block;
    a.per_xcd = (a.blocks_needed + 7) / 8;
    const int64_t grid = a.per_xcd * 8;
    if constexpr (EPL >= 100) {
        if constexpr (std::is_same<T, float>::value)
            k_apply_v4<G, EPL - 100, NOPS, NF, MODE><<<(unsigned)grid, block, 0, s>>>(a);
    } else {
        k_apply<T, G, EPL, NOPS, NF, MODE><<<(unsigned)grid, block, 0, s>>>(a);
    }
}

template <typename T, int G, int EPL, int MODE>
static bool dispatch_nops_nf(const ApplyArgs<T>& a, int nops, int nf, int block, hipStream_t s) {
    if (nf == 1) {
        switch (nops) {
            case 1: launch_apply<T, G, EPL, 1, 1, MODE>(a, block, s); return true;
            case 2: launch_apply<T, G, EPL, 2, 1, MODE>(a, block, s); return true;
            case 3: launch_apply<T, G, EPL, 3, 1, MODE>(a, block, s); return true;
            case 4: launch_apply<T, G, EPL, 4, 1, MODE>(a, block, s); return true;
        }
        return false;
    }
    if (nops != 1) return false;
    // fields per pass are capped at 32 / EPL (see max_fields) to bound registers
    switch (nf) {
        case 2: if constexpr (2 * (EPL >= 100 ? 4 * (EPL - 100) : EPL) <= 32) { launch_apply<T, G, EPL, 1, 2, MODE>(a, block, s); return true; }
                break;
        case 4: if constexpr (4 * (EPL >= 100 ? 4 * (EPL - 100) : EPL) <= 32) { launch_apply<T, G, EPL, 1, 4, MODE>(a, block, s); return true; }
                break;
        case 8: if constexpr (8 * (EPL >= 100 ? 4 * (EPL - 100) : EPL) <= 32) { launch_apply<T, G, EPL, 1, 8, MODE>(a, block, s); return true; }
                break;
        case 16: if constexpr (16 * (EPL >= 100 ? 4 * (EPL - 100) : EPL) <= 32) { launch_apply<T, G, EPL, 1, 16, MODE>(a, block, s); return true; }
                break;
    }
    return false;
}

// (lanes per row, elements per lane issued up front): every shape covers 64
// nonzeros per pass except the last two, which cover 128. Template EPL >= 100
// selects the 16-byte-load kernel with EPL - 100 chunks of 4 per lane.
template <typename T, int MODE>
static bool dispatch_group(const ApplyArgs<T>& a, int G, int epl, int nops, int nf, int block, hipStream_t s) {
    if (G == 4 && epl == 16) return dispatch_nops_nf<T, 4, 16, MODE>(a, nops, nf, block, s);
    if (G == 8 && epl == 8) return dispatch_nops_nf<T, 8, 8, MODE>(a, nops, nf, block, s);
    if (G == 16 && epl == 4) return dispatch_nops_nf<T, 16, 4, MODE>(a, nops, nf, block, s);
    if (G == 32 && epl == 2) return dispatch_nops_nf<T, 32, 2, MODE>(a, nops, nf, block, s);
    if (G == 64 && epl == 1) return dispatch_nops_nf<T, 64, 1, MODE>(a, nops, nf, block, s);
    if (G == 8 && epl == 16) return dispatch_nops_nf<T, 8, 16, MODE>(a, nops, nf, block, s);
    if (G == 16 && epl == 8) return dispatch_nops_nf<T, 16, 8, MODE>(a, nops, nf, block, s);
    return false;
}

// 16-byte-load shapes (FP32 only): epl = 4 * chunks per lane.
template <int MODE>
static bool dispatch_group_v4(const ApplyArgs<float>& a, int G, int epl, int nops, int nf, int block,
                              hipStream_t s) {
    if (G == 4 && epl == 8) return dispatch_nops_nf<float, 4, 102, MODE>(a, nops, nf, block, s);
    if (G == 8 && epl == 4) return dispatch_nops_nf<float, 8, 101, MODE>(a, nops, nf, block, s);
    if (G == 8 && epl == 8) return dispatch_nops_nf<float, 8, 102, MODE>(a, nops, nf, block, s);
    if (G == 8 && epl == 12) return dispatch_nops_nf<float, 8, 103, MODE>(a, nops, nf, block, s);
    if (G == 16 && epl == 4) return dispatch_nops_nf<float, 16, 101, MODE>(a, nops, nf, block, s);
    if (G == 16 && epl == 8) return dispatch_nops_nf<float, 16, 102, MODE>(a, nops, nf, block, s);
    if (G == 32 && epl == 4) return dispatch_nops_nf<float, 32, 101, MODE>(a, nops, nf, block, s);
    return false;
}

struct ApplyShape {
    int G, epl, vec;
    double mean;  // row length, 0: not looked up
};

// Launch shape from the mean row length (16-byte loads, 8 lanes per row): up
// to 24 nonzeros 4 per lane, up to 72 8 per lane, beyond 12 (rows of 93: one
// field 56 us against 47, 16 fields 255 against 205 with the strided tail from
// the 65th on, 343,000 rows; FP64 keeps 8). dcpse_set_apply_config overrides it.
static ApplyShape shape_of(dcpse_ctx* ctx, int64_t n_rows, int64_t nnz) {
    if (ctx->apply_group > 0) return {ctx->apply_group, ctx->apply_epl, ctx->apply_vec, 0.0};
    const double mean = n_rows > 0 ? (double)nnz / (double)n_rows : 0.0;
    return {8, mean <= 24 ? 4 : mean > 72 ? 12 : 8, 4, mean};
}

// The same where the caller gives no nnz: read once per (row_ptr, n_rows) and
// cached in the context, so repeated applies of one operator never synchronise
// the stream. (Another list at the same address, with as many rows, gets the
// shape of the first: another order of summation, and slower. The *_nnz entry
// points have no such memory.)
static ApplyShape auto_shape(dcpse_ctx* ctx, int64_t n_rows, const int64_t* row_ptr) {
    if (ctx->apply_group > 0) return {ctx->apply_group, ctx->apply_epl, ctx->apply_vec, 0.0};
    if (ctx->grp_rows == row_ptr && ctx->grp_n == n_rows) return {ctx->grp_g, ctx->grp_epl, ctx->grp_vec, ctx->grp_mean};
    int64_t nnz = 0;
    if (hipMemcpyAsync(&nnz, row_ptr + n_rows, sizeof(int64_t), hipMemcpyDeviceToHost, ctx->stream) != hipSuccess ||
        hipStreamSynchronize(ctx->stream) != hipSuccess)
        return {8, 8, 4, 0.0};  // not kept: the next call looks again
    const ApplyShape sh = shape_of(ctx, n_rows, nnz);
    ctx->grp_rows = row_ptr;
    ctx->grp_n = n_rows;
    ctx->grp_g = sh.G;
    ctx->grp_epl = sh.epl;
    ctx->grp_vec = sh.vec;
    ctx->grp_mean = sh.mean;
    return sh;
}

// Fields per pass: the largest compiled NF <= the remaining count and
// <= 32 / elems_per_lane (every field keeps EPL gathered values live).
static int field_chunk(int remaining, int nops, int epl) {
    if (nops != 1) return 1;
    const int cap = 32 / epl;
    for (int nf = 16; nf >= 2; nf >>= 1)
        if (remaining >= nf && nf <= cap) return nf;
    return 1;
}

// What a caller of the *_nnz entry points adds: the number of neighbours, which
// picks the launch shape, and device memory for the particle-major copies.
struct Counted {
    int64_t nnz;
    void* scratch;
    size_t bytes;
};

// Fields of a pass: the smallest of 4, 8 and 16 that holds nf.
static int pass_width(int nf) { return nf > 8 ? 16 : nf > 4 ? 8 : 4; }

template <typename T, int MODE>
static dcpse_status apply_impl(dcpse_ctx* ctx, int64_t n_rows, const int64_t* row_ptr, const int32_t* col,
                               int nops, const T* const* W, const T* f, int64_t ld_f, int nfields,
                               const T* f_self, int64_t ld_self, const T* diag, T* const* out, int64_t ld_out,
                               T alpha, T beta, const Counted* given = nullptr) {
    constexpr bool F32 = std::is_same<T, float>::value;
    if (!row_ptr || !col || !W || !f || !out || n_rows < 0 || nfields < 1 || nops < 1)
        return fail(ctx, DCPSE_ERR_INVALID, "null pointer or bad size");
    if (given && (given->nnz < 0 || (reinterpret_cast<uintptr_t>(given->scratch) & 15)))
        return fail(ctx, DCPSE_ERR_INVALID, "negative nnz or scratch not 16-byte aligned");
    if (nops > kMaxOps) return fail(ctx, DCPSE_ERR_UNSUPPORTED, "at most %d operators per pass", kMaxOps);
    if (nops > 1 && nfields > 1)
        return fail(ctx, DCPSE_ERR_UNSUPPORTED, "several operators and several fields in one pass");
    if (nfields > 1 && (ld_f < 1 || ld_out < n_rows || (f_self && ld_self < n_rows)))
        return fail(ctx, DCPSE_ERR_INVALID, "leading dimensions must cover the rows");
    for (int o = 0; o < nops; ++o)
        if (!W[o] || !out[o]) return fail(ctx, DCPSE_ERR_INVALID, "null operator pointer");
    if (n_rows == 0) return DCPSE_OK;
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    ApplyShape sh = given ? shape_of(ctx, n_rows, given->nnz) : auto_shape(ctx, n_rows, row_ptr);
    if (!F32 && ctx->apply_group <= 0 && sh.epl == 12) sh.epl = 8;
    const int block = ctx->apply_block;
    if (block % sh.G != 0 || block < 64 || block > kApplyMaxBlock)
        return fail(ctx, DCPSE_ERR_INVALID, "block %d incompatible with group %d", block, sh.G);
    ApplyArgs<T> a;
    a.n_rows = n_rows;
    a.row_ptr = row_ptr;
    a.col = col;
    a.diag = diag;
    a.ld_f = ld_f;
    a.ld_self = f_self ? ld_self : ld_f;
    a.ld_out = ld_out;
    a.alpha = alpha;
    a.beta = beta;
    for (int o = 0; o < kMaxOps; ++o) {
        a.W[o] = o < nops ? W[o] : nullptr;
        a.out[o] = nullptr;
    }
    int b0 = 0;
    // Batches of several fields on one set (no f_self: columns and rows index
    // the same n_rows particles; f_self == f may also be a domain that leads
    // its support set, with columns past the rows): interleaved up to 16 at a
    // time (the col/W streams read once per pass), the last ones in the
    // smallest of 4, 8 or 16 that holds them. The copy lies in the caller's
    // scratch, which a graph being captured may keep, or in the context's
    // workspace, which it may not (a later call can replace it): a captured
    // batch without scratch runs field by field, with the same bits.
    const bool particle_major = nops == 1 && nfields >= kBatchMin && !f_self &&
                                (F32 ? sh.vec == 4 && il_shape(sh.G, sh.epl) : ctx->apply_group <= 0);
    T* fil = nullptr;
    int width = 0;  // fields that the copy has room for
    std::optional<WorkspaceUse> use;
    if (particle_major && given) {
        const size_t room = given->scratch ? given->bytes / ((size_t)n_rows * sizeof(T)) : 0;
        fil = static_cast<T*>(given->scratch);
        width = room >= 16 ? 16 : room >= 8 ? 8 : room >= 4 ? 4 : 0;
    } else if (particle_major && !captured(ctx->stream)) {
        const size_t room = pass_width(nfields);
        Workspace ws;
        if (reserve_workspace(ctx, (size_t)n_rows * room * sizeof(T) + 256, &ws) == DCPSE_OK) {
            use.emplace(ctx);
            fil = ws.take<T>((size_t)n_rows * room);
            if (!fil) return fail(ctx, DCPSE_ERR_INVALID, "apply workspace sizing error");
            width = (int)room;
        }  // no room: field by field
    }
    while (width > 0 && nfields - b0 >= kBatchMin) {
        const int nf = std::min(nfields - b0, width), pass = pass_width(nf);
        const unsigned ib = (unsigned)((n_rows + 255) / 256);
        const T* fb = f + (int64_t)b0 * ld_f;
        if (pass == 16) k_interleave<16><<<ib, 256, 0, ctx->stream>>>(n_rows, fb, ld_f, nf, fil);
        else if (pass == 8) k_interleave<8><<<ib, 256, 0, ctx->stream>>>(n_rows, fb, ld_f, nf, fil);
        else k_interleave<4><<<ib, 256, 0, ctx->stream>>>(n_rows, fb, ld_f, nf, fil);
        DCPSE_LAUNCH_CHECK(ctx);
        a.f = a.f_self = fil;
        a.out[0] = out[0] + (int64_t)b0 * ld_out;
        bool ok = true;
        if constexpr (F32) {
            ok = pass == 16  ? dispatch_il<MODE, 16>(a, sh.G, sh.epl, nf, sh.mean, ctx->stream)
                 : pass == 8 ? dispatch_il<MODE, 8>(a, sh.G, sh.epl, nf, sh.mean, ctx->stream)
                             : dispatch_il<MODE, 4>(a, sh.G, sh.epl, nf, sh.mean, ctx->stream);
        } else {
            const int lanes = sh.epl == 4 ? 16 : 8;  // of the single-field kernel
            if (pass == 16) launch_batch64<16, MODE>(a, nf, lanes, ctx->stream);
            else if (pass == 8) launch_batch64<8, MODE>(a, nf, lanes, ctx->stream);
            else launch_batch64<4, MODE>(a, nf, lanes, ctx->stream);
        }
        if (!ok) return fail(ctx, DCPSE_ERR_UNSUPPORTED, "no batched apply kernel for group=%d x %d", sh.G, sh.epl);
        DCPSE_LAUNCH_CHECK(ctx);
        b0 += nf;
    }
    while (b0 < nfields) {
        const int nf = field_chunk(nfields - b0, nops, sh.epl);
        a.f = f + (int64_t)b0 * ld_f;
        a.f_self = (f_self ? f_self + (int64_t)b0 * ld_self : a.f);
        for (int o = 0; o < nops; ++o) a.out[o] = out[o] + (int64_t)b0 * ld_out;
        bool ok = false;
        if constexpr (std::is_same<T, float>::value)
            ok = sh.vec == 4 ? dispatch_group_v4<MODE>(a, sh.G, sh.epl, nops, nf, block, ctx->stream)
                             : dispatch_group<T, MODE>(a, sh.G, sh.epl, nops, nf, block, ctx->stream);
        else
            ok = dispatch_group<T, MODE>(a, sh.G, sh.epl, nops, nf, block, ctx->stream) ||
                 (sh.vec == 4 && dispatch_group<T, MODE>(a, 16, 4, nops, nf, block, ctx->stream));
        if (!ok)
            return fail(ctx, DCPSE_ERR_UNSUPPORTED, "no apply kernel for group=%d x %d ops=%d fields=%d", sh.G,
                        sh.epl, nops, nf);
        DCPSE_LAUNCH_CHECK(ctx);
        b0 += nf;
    }
    return DCPSE_OK;
}

// y = alpha * x + beta * y (beta == 0 never reads y)
template <typename T>
__global__ void k_axpby(int64_t n, T alpha, const T* __restrict__ x, T beta, T* __restrict__ y) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        y[i] = beta != T(0) ? fma(alpha, x[i], beta * y[i]) : alpha * x[i];
}

template <typename T>
static dcpse_status axpby(dcpse_ctx* ctx, int64_t n, T alpha, const T* x, T beta, T* y) {
    if (!ctx) return DCPSE_ERR_INVALID;
    if (n < 0 || (n > 0 && (!x || !y))) return fail(ctx, DCPSE_ERR_INVALID, "null pointer or negative size");
    DCPSE_HIP_CHECK(ctx, hipSetDevice(ctx->device));
    if (n == 0) return DCPSE_OK;
    const int64_t b = std::min<int64_t>((n + 255) / 256, (int64_t)ctx->num_cus * 8);
    k_axpby<T><<<(unsigned)b, 256, 0, ctx->stream>>>(n, alpha, x, beta, y);
    DCPSE_LAUNCH_CHECK(ctx);
    return DCPSE_OK;
}

}  // namespace dcpse

using namespace dcpse;

extern "C" {

dcpse_status dcpse_apply_f32(dcpse_ctx* ctx, int64_t n_rows, const int64_t* row_ptr, const int32_t* col,
                             int32_t n_ops, const float* const* W, const float* f, int64_t ld_f, int32_t n_fields,
                             const float* f_self, int64_t ld_self, float* const* out, int64_t ld_out, float alpha,
                             float beta) {
    if (!ctx) return DCPSE_ERR_INVALID;
    return apply_impl<float, kDiff>(ctx, n_rows, row_ptr, col, n_ops, W, f, ld_f, n_fields, f_self, ld_self,
                                    nullptr, out, ld_out, alpha, beta);
}

dcpse_status dcpse_apply_f64(dcpse_ctx* ctx, int64_t n_rows, const int64_t* row_ptr, const int32_t* col,
                             int32_t n_ops, const double* const* W, const double* f, int64_t ld_f,
                             int32_t n_fields, const double* f_self, int64_t ld_self, double* const* out,
                             int64_t ld_out, double alpha, double beta) {
    if (!ctx) return DCPSE_ERR_INVALID;
    return apply_impl<double, kDiff>(ctx, n_rows, row_ptr, col, n_ops, W, f, ld_f, n_fields, f_self, ld_self,
                                     nullptr, out, ld_out, alpha, beta);
}

dcpse_status dcpse_apply_transpose_f32(dcpse_ctx* ctx, int64_t n_cols, const int64_t* rowT_ptr,
                                       const int32_t* colT, const float* WT, const float* diag, const float* g,
                                       int64_t ld_g, int32_t n_fields, float* out, int64_t ld_out, float alpha,
                                       float beta) {
    if (!ctx) return DCPSE_ERR_INVALID;
    if (!diag) return fail(ctx, DCPSE_ERR_INVALID, "diag is null");
    const float* Wp[1] = {WT};
    float* Op[1] = {out};
    return apply_impl<float, kExplicitDiag>(ctx, n_cols, rowT_ptr, colT, 1, Wp, g, ld_g, n_fields, nullptr, ld_g,
                                            diag, Op, ld_out, alpha, beta);
}

dcpse_status dcpse_apply_transpose_f64(dcpse_ctx* ctx, int64_t n_cols, const int64_t* rowT_ptr,
                                       const int32_t* colT, const double* WT, const double* diag,
                                       const double* g, int64_t ld_g, int32_t n_fields, double* out,
                                       int64_t ld_out, double alpha, double beta) {
    if (!ctx) return DCPSE_ERR_INVALID;
    if (!diag) return fail(ctx, DCPSE_ERR_INVALID, "diag is null");
    const double* Wp[1] = {WT};
    double* Op[1] = {out};
    return apply_impl<double, kExplicitDiag>(ctx, n_cols, rowT_ptr, colT, 1, Wp, g, ld_g, n_fields, nullptr, ld_g,
                                             diag, Op, ld_out, alpha, beta);
}

dcpse_status dcpse_apply_nnz_f32(dcpse_ctx* ctx, int64_t n_rows, int64_t nnz, const int64_t* row_ptr,
                                 const int32_t* col, int32_t n_ops, const float* const* W, const float* f, int64_t ld_f,
                                 int32_t n_fields, const float* f_self, int64_t ld_self, float* const* out,
                                 int64_t ld_out, float alpha, float beta, void* scratch, size_t scratch_bytes) {
    if (!ctx) return DCPSE_ERR_INVALID;
    const Counted given{nnz, scratch, scratch_bytes};
    return apply_impl<float, kDiff>(ctx, n_rows, row_ptr, col, n_ops, W, f, ld_f, n_fields, f_self, ld_self, nullptr,
                                  out, ld_out, alpha, beta, &given);
}

dcpse_status dcpse_apply_transpose_nnz_f32(dcpse_ctx* ctx, int64_t n_cols, int64_t nnz, const int64_t* rowT_ptr,
                                           const int32_t* colT, const float* WT, const float* diag, const float* g,
                                           int64_t ld_g, int32_t n_fields, float* out, int64_t ld_out, float alpha,
                                           float beta, void* scratch, size_t scratch_bytes) {
    if (!ctx) return DCPSE_ERR_INVALID;
    if (!diag) return fail(ctx, DCPSE_ERR_INVALID, "diag is null");
    const float* Wp[1] = {WT};
    float* Op[1] = {out};
    const Counted given{nnz, scratch, scratch_bytes};
    return apply_impl<float, kExplicitDiag>(ctx, n_cols, rowT_ptr, colT, 1, Wp, g, ld_g, n_fields, nullptr, ld_g, diag,
                                          Op, ld_out, alpha, beta, &given);
}

dcpse_status dcpse_apply_nnz_f64(dcpse_ctx* ctx, int64_t n_rows, int64_t nnz, const int64_t* row_ptr,
                                 const int32_t* col, int32_t n_ops, const double* const* W, const double* f, int64_t ld_f,
                                 int32_t n_fields, const double* f_self, int64_t ld_self, double* const* out,
                                 int64_t ld_out, double alpha, double beta, void* scratch, size_t scratch_bytes) {
    if (!ctx) return DCPSE_ERR_INVALID;
    const Counted given{nnz, scratch, scratch_bytes};
    return apply_impl<double, kDiff>(ctx, n_rows, row_ptr, col, n_ops, W, f, ld_f, n_fields, f_self, ld_self, nullptr,
                                  out, ld_out, alpha, beta, &given);
}

dcpse_status dcpse_apply_transpose_nnz_f64(dcpse_ctx* ctx, int64_t n_cols, int64_t nnz, const int64_t* rowT_ptr,
                                           const int32_t* colT, const double* WT, const double* diag, const double* g,
                                           int64_t ld_g, int32_t n_fields, double* out, int64_t ld_out, double alpha,
                                           double beta, void* scratch, size_t scratch_bytes) {
    if (!ctx) return DCPSE_ERR_INVALID;
    if (!diag) return fail(ctx, DCPSE_ERR_INVALID, "diag is null");
    const double* Wp[1] = {WT};
    double* Op[1] = {out};
    const Counted given{nnz, scratch, scratch_bytes};
    return apply_impl<double, kExplicitDiag>(ctx, n_cols, rowT_ptr, colT, 1, Wp, g, ld_g, n_fields, nullptr, ld_g, diag,
                                          Op, ld_out, alpha, beta, &given);
}

dcpse_status dcpse_axpby_f32(dcpse_ctx* ctx, int64_t n, float alpha, const float* x, float beta, float* y) {
    return axpby<float>(ctx, n, alpha, x, beta, y);
}

dcpse_status dcpse_axpby_f64(dcpse_ctx* ctx, int64_t n, double alpha, const double* x, double beta, double* y) {
    return axpby<double>(ctx, n, alpha, x, beta, y);
}

}  // extern "C"
