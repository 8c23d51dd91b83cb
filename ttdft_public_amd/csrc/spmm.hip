// Hamiltonian application kernels: H X = H_loc X + C^T (D C X), with the
// three-term Chebyshev recurrence fused into the SpMM epilogue.
//
// Data layout: X, Y are basis-major blocks (X[i*ld + j], state j of basis
// function i), so one H_loc row reads whole contiguous state rows of X and a
// 64-wide wavefront loads 64 consecutive states of one basis function in one
// coalesced access.  One wavefront owns one H_loc row and all k states
// (NC = ceil(k/64) accumulator chunks per lane), so H_loc is streamed from
// HBM exactly once per application; the row's (value, column) pairs are read
// 64 at a time with one coalesced load and broadcast with v_readlane.
#include <algorithm>

#include "internal.h"
#include "lds_ring.h"

namespace ttdft {
namespace {

__device__ __forceinline__ double bcast(double v, int l) {
    const long long b = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ float bcast(float v, int l) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l));
}
__device__ __forceinline__ int bcast(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

template <typename T, int NC>
__global__ __launch_bounds__(256) void spmm_fused_kernel(
    int64_t n, const int64_t *__restrict__ rowptr, const int32_t *__restrict__ col,
    const T *__restrict__ val, const T *__restrict__ X, int64_t ldx,
    const int64_t *__restrict__ ct_rowptr, const int32_t *__restrict__ ct_col,
    const T *__restrict__ ct_val, const T *__restrict__ W, int32_t ldw, T *Y, int64_t ldy,
    const T *Z, int64_t ldz, int32_t k, T alpha, T beta, T delta, int use_beta,
    int use_delta) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (row >= n) return;
    T acc[NC];
#pragma unroll
    for (int t = 0; t < NC; ++t) acc[t] = T(0);

    // U nonzeros per step: their X rows are loaded together before the
    // multiply-adds, so a wave keeps U gathers in flight instead of one (the
    // adds still run in the row's order).  Lanes past the chunk's count hold
    // value 0 and column 0, so the last step reads row 0 and adds zeros.
    constexpr int U = NC <= 2 ? 8 : (NC <= 4 ? 4 : 2);
    const int64_t e0 = rowptr[row], e1 = rowptr[row + 1];
    for (int64_t base = e0; base < e1; base += 64) {
        const int cnt = (int)((e1 - base) < 64 ? (e1 - base) : 64);
        T v = T(0);
        int c = 0;
        if (lane < cnt) {
            v = val[base + lane];
            c = col[base + lane];
        }
        const int steps = (cnt + U - 1) / U;
        for (int s = 0; s < steps; ++s) {
            T a[U], xv[U][NC];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                a[u] = bcast(v, s * U + u);
                const T *xr = X + (int64_t)bcast(c, s * U + u) * ldx + lane;
#pragma unroll
                for (int t = 0; t < NC; ++t) xv[u][t] = lane + 64 * t < k ? xr[64 * t] : T(0);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int t = 0; t < NC; ++t) acc[t] += a[u] * xv[u][t];
        }
    }
    if (ct_rowptr != nullptr) {
        const int64_t f0 = ct_rowptr[row], f1 = ct_rowptr[row + 1];
        for (int64_t e = f0; e < f1; ++e) {
            const T a = ct_val[e];
            const T *wr = W + (int64_t)ct_col[e] * ldw + lane;
#pragma unroll
            for (int t = 0; t < NC; ++t) {
                if (lane + 64 * t < k) acc[t] += a * wr[64 * t];
            }
        }
    }
    T *yr = Y + row * ldy + lane;
    const T *xr = X + row * ldx + lane;
    const T *zr = Z + row * ldz + lane;
#pragma unroll
    for (int t = 0; t < NC; ++t) {
        if (lane + 64 * t < k) {
            T y = acc[t] * alpha;
            if (use_beta) y = y + beta * xr[64 * t];
            if (use_delta) y = y + delta * zr[64 * t];
            yr[64 * t] = y;
        }
    }
}

// Single-vector H_loc application for the Lanczos bound estimator:
// y = H_loc x + C^T w.  One wavefront per row; lanes stride over the row's
// nonzeros (coalesced value/index loads, gathered x) and the partial sums are
// combined with a wavefront shuffle reduction.
__global__ __launch_bounds__(256) void spmv_kernel(
    int64_t n, const int64_t *__restrict__ rowptr, const int32_t *__restrict__ col,
    const double *__restrict__ val, const double *__restrict__ x,
    const int64_t *__restrict__ ct_rowptr, const int32_t *__restrict__ ct_col,
    const double *__restrict__ ct_val, const double *__restrict__ w, double *__restrict__ y) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n) return;
    double s = 0.0;
    for (int64_t e = rowptr[row] + lane; e < rowptr[row + 1]; e += 64) s += val[e] * x[col[e]];
    if (ct_rowptr)
        for (int64_t e = ct_rowptr[row] + lane; e < ct_rowptr[row + 1]; e += 64)
            s += ct_val[e] * w[ct_col[e]];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) y[row] = s;
}

// W[r][j] = sum_e (D C)[r][e] X[col_e][j].  A projector row has a few
// thousand nonzeros and there are only a few hundred rows, so one block per
// row would leave most CUs idle: block (r, panel, split) takes 64 states and
// one of nsplit slices of row r's nonzeros (4 wavefronts over the slice,
// summed through LDS) and writes a partial sum; nl_reduce_kernel adds the
// nsplit partials in a fixed order (deterministic).  X rows are gathered 8 at
// a time so their loads are in flight together.
template <typename T>
__global__ __launch_bounds__(256) void nl_project_kernel(
    int32_t p, int32_t npanel, int32_t nsplit, const int64_t *__restrict__ c_rowptr,
    const int32_t *__restrict__ c_col, const T *__restrict__ c_val, const T *__restrict__ X,
    int64_t ldx, int32_t k, T *__restrict__ Wp) {
    __shared__ T red[4][64];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    int b = blockIdx.x;
    const int split = b % nsplit;
    b /= nsplit;
    const int panel = b % npanel;
    const int r = b / npanel;
    const int c = panel * 64 + lane;
    const int cc = c < k ? c : k - 1;  // clamped: every lane loads a valid element
    const int64_t e0 = c_rowptr[r], len = c_rowptr[r + 1] - e0;
    const int64_t lo = e0 + len * split / nsplit, hi = e0 + len * (split + 1) / nsplit;
    T acc = T(0);
    for (int64_t base = lo + 64 * wave; base < hi; base += 256) {
        const int cnt = (int)((hi - base) < 64 ? (hi - base) : 64);
        T v = T(0);
        int col = 0;
        if (lane < cnt) {
            v = c_val[base + lane];
            col = c_col[base + lane];
        }
        int j = 0;
        for (; j + 8 <= cnt; j += 8) {
            T x[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) x[u] = X[(int64_t)bcast(col, j + u) * ldx + cc];
#pragma unroll
            for (int u = 0; u < 8; ++u) acc += bcast(v, j + u) * x[u];
        }
        for (; j < cnt; ++j) acc += bcast(v, j) * X[(int64_t)bcast(col, j) * ldx + cc];
    }
    red[wave][lane] = acc;
    __syncthreads();
    if (wave == 0 && c < k)
        Wp[((int64_t)split * p + r) * k + c] =
            (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]);
}

template <typename T>
__global__ void nl_reduce_kernel(int64_t pk, int32_t nsplit, const T *__restrict__ Wp,
                                 T *__restrict__ W) {
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < pk;
         e += (int64_t)gridDim.x * blockDim.x) {
        T s = Wp[e];
        for (int q = 1; q < nsplit; ++q) s += Wp[(int64_t)q * pk + e];
        W[e] = s;
    }
}

// slices per projector row: about 4096 blocks in all, at least 256 nonzeros a slice
int nl_splits(const ttdft_ham_s *H, int32_t k) {
    if (H->p == 0) return 1;
    const int64_t npanel = (k + 63) / 64;
    int64_t ns = (4096 + H->p * npanel - 1) / (H->p * npanel);
    const int64_t cap = H->nnz_c / H->p / 256;
    if (ns > cap) ns = cap;
    if (ns < 1) ns = 1;
    if (ns > 64) ns = 64;
    return (int)ns;
}

template <typename T>
int nl_launch(ttdft_ctx ctx, const ttdft_ham_s *H, const T *X, int64_t ldx, int32_t k,
              const T *c_val, T *W) {
    const int npanel = (k + 63) / 64;
    const int ns = nl_splits(H, k);
    T *Wp = ns > 1 ? W + (int64_t)H->p * k : W;
    hipLaunchKernelGGL(nl_project_kernel<T>, dim3((unsigned)((int64_t)H->p * npanel * ns)),
                       dim3(256), 0, ctx->stream, H->p, npanel, ns, H->c_rowptr, H->c_col, c_val,
                       X, ldx, k, Wp);
    TT_LAUNCH_CHECK();
    if (ns > 1) {
        const int64_t pk = (int64_t)H->p * k;
        int64_t blocks = (pk + 255) / 256;
        if (blocks > 4096) blocks = 4096;
        hipLaunchKernelGGL(nl_reduce_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, ctx->stream,
                           pk, ns, Wp, W);
        TT_LAUNCH_CHECK();
    }
    return TTDFT_OK;
}

// D[row][col_e] = val_e (D zeroed beforehand, leading dimension ld); one
// wavefront per row
template <typename T>
__global__ __launch_bounds__(256) void csr_to_dense_kernel(int64_t n, int64_t ld,
                                                           const int64_t *__restrict__ rowptr,
                                                           const int32_t *__restrict__ col,
                                                           const T *__restrict__ val,
                                                           T *__restrict__ D) {
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n) return;
    for (int64_t e = rowptr[row] + lane; e < rowptr[row + 1]; e += 64)
        D[row * ld + col[e]] = val[e];
}

// Dense H_loc X with the recurrence epilogue, on matrix cores: a workgroup
// owns 16 rows of Y and 16 JT states; its 8 waves split the inner dimension l
// in eight and their partial tiles are summed through LDS.
//
// Storage: row-major, leading dimension ldh = n rounded up to 32, rows padded
// to a multiple of 16, padding zero.  Per 32-wide step of l, lane (i, q)
// (i = lane % 16, q = lane / 16) loads the 8 consecutive entries
// H[i0 + i][l0 + 8q .. 8q + 7] with wide loads, so each row of the tile is one
// contiguous 32-entry run, and the 8 matching rows of X; MFMA step u
// (u = 0..7) then pairs l = l0 + 8q + u in both operands.  The next step's
// loads are issued before this step's products (two register buffers).  X
// rows past n are read clamped to row n - 1 (finite values times the zero
// padding) and states past k clamped to k - 1 (never stored), so no load is
// predicated.
//
// The product is D[j][i] = sum_l X[l][j] H[i][l]: A operand X^T (16 states x
// 4 l, lane j + 16 kk), B operand H^T (4 l x 16 rows, lane i + 16 kk).  FP64
// storage runs on 16x16x4 FP64 MFMA (element v of lane L is D[L/16 + 4v][L%16])
// and FP32 storage on 16x16x4 FP32 MFMA with FP32 accumulation (element v of
// lane L is D[4 (L/16) + v][L%16]).  Then
// Y[i][j] = alpha (HX[i][j] + sum_e ct[e] W[ct_col_e][j]) (+ beta X[i][j]) (+ delta Z[i][j]).
typedef double dv4 __attribute__((ext_vector_type(4)));
typedef float fv4 __attribute__((ext_vector_type(4)));
constexpr int kDenseWaves = 8;

template <typename T> struct DenseMma;
template <> struct DenseMma<double> {
    typedef dv4 acc_t;
    static __device__ __forceinline__ dv4 step(double a, double b, dv4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int state(int q, int v) { return q + 4 * v; }
};
template <> struct DenseMma<float> {
    typedef fv4 acc_t;
    static __device__ __forceinline__ fv4 step(float a, float b, fv4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int state(int q, int v) { return 4 * q + v; }
};

// Stage depth U (MFMA steps per stage, U consecutive entries per lane) and
// accumulator sets NA per state-tile count: up to 64 states, 8-deep stages and
// two accumulator sets (alternate steps); 80 or 96 states, 4-deep stages and
// one set, which keeps the two stages in registers.
template <int JT> struct DenseCfg {
    static constexpr int U = JT <= 4 ? 8 : 4;
    static constexpr int NA = JT <= 4 ? 2 : 1;
};

template <typename T, int JT> struct DenseStage {
    static constexpr int U = DenseCfg<JT>::U;
    T h[U];
    T x[U][JT];
};

template <typename T, int JT, bool CONTIG>
__device__ __forceinline__ void dense_load(DenseStage<T, JT> &st, const T *hrow, const T *X,
                                           int64_t ldx, int64_t n, const int *cidx, int64_t l0,
                                           int q) {
    constexpr int U = DenseCfg<JT>::U;
    // U consecutive entries (16-64 B), aligned by the padding
    typedef T vU __attribute__((ext_vector_type(U)));
    typedef T v2 __attribute__((ext_vector_type(2)));
    const vU hv = *reinterpret_cast<const vU *>(hrow + l0);
#pragma unroll
    for (int u = 0; u < U; ++u) st.h[u] = hv[u];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        int64_t l = l0 + U * q + u;
        l = l < n ? l : n - 1;
        const T *xr = X + l * ldx;
        if constexpr (CONTIG) {
            // the lane's JT states are consecutive from cidx[0] (even, with
            // ldx even): pairs in one load each
#pragma unroll
            for (int jt = 0; jt < JT; jt += 2) {
                const v2 w = *reinterpret_cast<const v2 *>(xr + cidx[0] + jt);
                st.x[u][jt] = w[0];
                st.x[u][jt + 1] = w[1];
            }
        } else {
#pragma unroll
            for (int jt = 0; jt < JT; ++jt) st.x[u][jt] = xr[cidx[jt]];
        }
    }
}

template <typename T, int JT>
__device__ __forceinline__ void dense_mma(
    const DenseStage<T, JT> &st, typename DenseMma<T>::acc_t (&acc)[DenseCfg<JT>::NA][JT]) {
    constexpr int U = DenseCfg<JT>::U, NA = DenseCfg<JT>::NA;
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
        for (int jt = 0; jt < JT; ++jt)
            acc[u % NA][jt] = DenseMma<T>::step(st.x[u][jt], st.h[u], acc[u % NA][jt]);
}

template <typename T, int JT, bool CONTIG>
__global__ __launch_bounds__(512) void dense_hx_kernel(
    int64_t n, int64_t ldh, int32_t k, const T *__restrict__ H, const T *X, int64_t ldx,
    const int64_t *__restrict__ ct_rowptr, const int32_t *__restrict__ ct_col,
    const T *__restrict__ ct_val, const T *__restrict__ W, T *Y, int64_t ldy, const T *Z,
    int64_t ldz, double alpha, double beta, double delta, int use_beta, int use_delta) {
    typedef typename DenseMma<T>::acc_t acc_t;
    constexpr int U = DenseCfg<JT>::U, NA = DenseCfg<JT>::NA, SW = 4 * U;  // step width in l
    __shared__ T red[kDenseWaves][16 * JT][17];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int li = lane & 15, q = lane >> 4;
    const int64_t i0 = (int64_t)blockIdx.x * 16;
    const int c0 = blockIdx.y * 16 * JT;
    const int64_t part = ((ldh + kDenseWaves - 1) / kDenseWaves + SW - 1) / SW * SW;
    const int64_t lb = wave * part, le = lb + part < ldh ? lb + part : ldh;
    const T *hrow = H + (i0 + li) * ldh + U * q;
    // state of tile jt, tile row i: c0 + 16 jt + i, or with CONTIG (every tile
    // full, ldx even) c0 + JT i + jt, so a lane's JT states are consecutive
    int cidx[JT];
#pragma unroll
    for (int jt = 0; jt < JT; ++jt) {
        const int c = CONTIG ? c0 + JT * li + jt : c0 + 16 * jt + li;
        cidx[jt] = c < k ? c : k - 1;
    }
    acc_t acc[NA][JT];
#pragma unroll
    for (int e = 0; e < NA; ++e)
#pragma unroll
        for (int jt = 0; jt < JT; ++jt) acc[e][jt] = acc_t{0, 0, 0, 0};
    if (lb < le) {
        // two buffers, the loads of step s + 1 in flight during the products
        // of step s (the last pair reloads the final step into the idle
        // buffer; scheduling barriers keep the compiler from sinking the loads
        // into the products)
        DenseStage<T, JT> sa, sb;
        const int64_t nsteps = (le - lb) / SW;
        dense_load<T, JT, CONTIG>(sa, hrow, X, ldx, n, cidx, lb, q);
        int64_t st = 0;
        for (; st + 2 <= nsteps; st += 2) {
            dense_load<T, JT, CONTIG>(sb, hrow, X, ldx, n, cidx, lb + SW * (st + 1), q);
            __builtin_amdgcn_sched_barrier(0);
            dense_mma<T, JT>(sa, acc);
            __builtin_amdgcn_sched_barrier(0);
            const int64_t s2 = st + 2 < nsteps ? st + 2 : nsteps - 1;
            dense_load<T, JT, CONTIG>(sa, hrow, X, ldx, n, cidx, lb + SW * s2, q);
            __builtin_amdgcn_sched_barrier(0);
            dense_mma<T, JT>(sb, acc);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (st < nsteps) dense_mma<T, JT>(sa, acc);
    }
#pragma unroll
    for (int jt = 0; jt < JT; ++jt)
#pragma unroll
        for (int v = 0; v < 4; ++v)
            red[wave][16 * jt + DenseMma<T>::state(q, v)][li] =
                NA == 2 ? acc[0][jt][v] + acc[NA - 1][jt][v] : acc[0][jt][v];
    __syncthreads();
    for (int e = t; e < 16 * 16 * JT; e += 512) {
        const int j = e % (16 * JT), ii = e / (16 * JT);
        const int64_t r = i0 + ii;
        const int c = CONTIG ? c0 + JT * (j % 16) + j / 16 : c0 + j;
        if (r >= n || c >= k) continue;
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < kDenseWaves; ++w) s += (double)red[w][j][ii];
        if (ct_rowptr)
            for (int64_t f = ct_rowptr[r]; f < ct_rowptr[r + 1]; ++f)
                s += (double)ct_val[f] * (double)W[(int64_t)ct_col[f] * k + c];
        double y = s * alpha;
        if (use_beta) y += beta * (double)X[r * ldx + c];
        if (use_delta) y += delta * (double)Z[r * ldz + c];
        Y[r * ldy + c] = (T)y;
    }
}

// Dense H_loc X through a ring of LDS stages, in two or three kernels.
//
// What bounds it: H is read once per product and fits no cache, so HBM does
// (6.1 TB/s for a plain read), beside the matrix cores in FP64 from about 64
// states on.  dense_ring_kernel therefore keeps two further stages of loads in
// flight while one is multiplied: workgroup (row block, state block, part)
// owns ROWS rows (8 waves of 16 in FP64, of 32 in FP32) by 16 JT states over
// part p of the inner dimension l.  A stage is 32 values of l: 32 KB of H,
// each wave its own rows, loaded straight into LDS 16 bytes a lane in whole
// row runs; and the same 32 rows of X, shared by the waves.  One barrier per
// stage.  The 16-byte chunks of an H row are stored at (chunk ^ row), so that
// the operand reads of 16 rows spread over the banks.
//
// X comes as MFMA fragments (layout below; 1 KB pieces that are loaded and
// read lane-contiguous), made by x_fragments_kernel or, within a filter, by
// dense_combine_kernel as it writes the previous product's result.
//
// FP64: D[j][i] = sum_l X[l][j] H[i][l] on 16x16x4 FP64 MFMA.
//
// FP32: FP32 MFMA has a sixteenth of the BF16 rate and bounded this product
// (27,000 x 96: 1.33 ms where the read of H takes 0.48).  Every FP32 value is
// the exact sum of three BF16 values (x0 = bf16(x), x1 = bf16(x - x0),
// x2 = x - x0 - x1); the products h0 x0, h0 x1, h1 x0, h1 x1, h0 x2, h2 x0
// on 16x16x32 BF16 MFMA with FP32 accumulation leave out terms below 2^-24 of
// |h x|, the rounding of one FP32 product.  H stays in FP32 in memory and is
// split in registers after the LDS read, X once per product, times 2^16 so that
// the third piece of every normal number is one too (H's entries keep their 24
// bits from 2^-110 on).  A value that the pieces cannot hold (infinities, X from
// 2^111 on) makes the sum infinite or NaN; dense_combine_kernel then adds up that
// row again in plain FP32.
//
// dense_combine_kernel: Y = alpha (sum_p P[p] + C^T W) (+ beta X) (+ delta Z),
// the parts summed in FP64 in a fixed order.
constexpr int kRingStep = 32;  // values of l per stage

typedef __bf16 bfv8 __attribute__((ext_vector_type(8)));
typedef unsigned uv4 __attribute__((ext_vector_type(4)));

// Fragments of 32 rows of X and one 16-state tile, lane = state + 16 q:
//   FP64: four 1 KB pieces u2 of two doubles per lane, X[8 u2 + 2 q + {0, 1}];
//   FP32: three 1 KB pieces (x0, x1, x2) of eight BF16 per lane, X[8 q + 0..7].
// Pieces of one tile are consecutive, then tiles, then steps.
template <typename T> struct RingCfg;
template <> struct RingCfg<double> {
    static constexpr int RT = 1;      // 16-row tiles per wave
    static constexpr int PIECES = 4;  // 1 KB pieces per tile and step
};
template <> struct RingCfg<float> {
    static constexpr int RT = 2;
    static constexpr int PIECES = 3;
};
constexpr int kRingWaves = 8;
template <typename T> constexpr int ring_rows() { return 16 * kRingWaves * RingCfg<T>::RT; }

// Two FP32 values as sums of three BF16 values each, packed in pairs.
__device__ __forceinline__ unsigned bf16_pair(float x, float y) {
    typedef float v2 __attribute__((ext_vector_type(2)));
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v2{x, y}, b2));
}
__device__ __forceinline__ void split_bf16(float x, float y, unsigned &a, unsigned &b,
                                           unsigned &c) {
    a = bf16_pair(x, y);
    const float rx = x - __builtin_bit_cast(float, a << 16);
    const float ry = y - __builtin_bit_cast(float, a & 0xffff0000u);
    b = bf16_pair(rx, ry);
    c = bf16_pair(rx - __builtin_bit_cast(float, b << 16),
                  ry - __builtin_bit_cast(float, b & 0xffff0000u));
}

// Factor of the FP32 fragments, undone where their sums are complete
constexpr float kFragScale = 65536.0f;

// Sign that FP32 fragments of stage `st` carry in state c, undone as the
// stage's sums are added up: (-1)^c times stage_sign.  A BF16 product rounds
// its aligned terms towards minus infinity, so without it every sum of small
// terms would err to the same side; a filter adds that up over its steps
// (8,000 x 24, degree 20: error 1.2e-5 in place of 1.0e-6; FP32 products 4.9e-6).
__device__ __forceinline__ unsigned stage_flip(int64_t st) {
    return ((unsigned)st * 2654435761u) & 0x80000000u;
}

// Writes the fragment entries of rows 8 o .. 8 o + 7 of state c.
__device__ __forceinline__ void store_fragment(const double (&y)[8], int64_t o, int c,
                                               int32_t ntiles, double *F) {
    typedef double v2 __attribute__((ext_vector_type(2)));
    double *f = F + (((o >> 2) * ntiles + (c >> 4)) * 4 + (o & 3)) * 128 + 2 * (c & 15);
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<v2 *>(f + 32 * q) = v2{y[2 * q], y[2 * q + 1]};
}
__device__ __forceinline__ void store_fragment(const float (&y)[8], int64_t o, int c,
                                               int32_t ntiles, float *F) {
    uv4 a, b, d;
    const float scale =
        __builtin_bit_cast(float, __builtin_bit_cast(unsigned, kFragScale) ^ stage_flip(o >> 2) ^
                                      ((unsigned)(c & 1) << 31));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        unsigned p, q, r;
        split_bf16(y[2 * i] * scale, y[2 * i + 1] * scale, p, q, r);
        a[i] = p;
        b[i] = q;
        d[i] = r;
    }
    // (a piece is 64 lanes x 16 bytes)
    uv4 *f = reinterpret_cast<uv4 *>(F) + ((o >> 2) * ntiles + (c >> 4)) * 3 * 64 + (c & 15) +
             16 * (o & 3);
    f[0] = a;
    f[64] = b;
    f[128] = d;
}

// X to fragments: one thread per eight rows of one state; rows n .. ldh - 1
// are zero (they meet the zero padding of H), states past k are left as they
// are (they only reach results that are not stored).
template <typename T>
__global__ __launch_bounds__(256) void x_fragments_kernel(int64_t n, int64_t ldh, int32_t k,
                                                          const T *__restrict__ X, int64_t ldx,
                                                          int32_t ntiles, T *__restrict__ F) {
    const unsigned e = blockIdx.x * 256u + threadIdx.x;
    const unsigned oc = e / (unsigned)k;
    const int c = (int)(e - oc * (unsigned)k);
    const int64_t o = oc;
    if (o >= ldh / 8) return;
    T y[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = 8 * o + i < n ? X[(8 * o + i) * ldx + c] : T(0);
    store_fragment(y, o, c, ntiles, F);
}

// A wave's H operands of one stage in registers
template <typename T> struct RingH;
template <> struct RingH<double> {
    v4f_t raw[4];
    __device__ __forceinline__ void read(const unsigned char *hb, int wave, int lane) {
        const int li = lane & 15, q = lane >> 4;
        // row li of the wave's tile, chunk 4 u2 + q at position (4 u2 + q) ^ li
        const unsigned a = lds_addr(hb) + (16 * wave + li) * 256 + ((q ^ li) * 16);
        lds_read4(a, a ^ 64, a ^ 128, a ^ 192, raw[0], raw[1], raw[2], raw[3]);
    }
    __device__ __forceinline__ void split(int, int) {}
};
template <> struct RingH<float> {
    v4f_t raw[4];
    uv4 h0[2], h1[2], h2[2];  // BF16 pieces of rows li, li + 16
    __device__ __forceinline__ void read(const unsigned char *hb, int wave, int lane) {
        const int li = lane & 15, q = lane >> 4;
        // rows li and li + 16 of the wave, chunks 2 q and 2 q + 1 (entries 8 q .. 8 q + 7)
        const unsigned a = lds_addr(hb) + (32 * wave + li) * 128 + (((2 * q) ^ (li & 7)) * 16);
        lds_read4(a, a ^ 16, a + 2048, (a ^ 16) + 2048, raw[0], raw[1], raw[2], raw[3]);
    }
    // pairs lo .. hi - 1 of the lane's eight
    __device__ __forceinline__ void split(int lo, int hi) {
#pragma unroll
        for (int e = lo; e < hi; ++e) {
            unsigned a, b, c;
            split_bf16(raw[e >> 1][2 * (e & 1)], raw[e >> 1][2 * (e & 1) + 1], a, b, c);
            // (pins the conversion here: it would sink past the stage's barrier)
            asm volatile("" : "+v"(a), "+v"(b), "+v"(c));
            h0[e >> 2][e & 3] = a;
            h1[e >> 2][e & 3] = b;
            h2[e >> 2][e & 3] = c;
        }
    }
};

// Products of one stage.  While they run, `next` reads (and splits) the H
// operands of the stage after: all waves leave the stage's barrier together,
// and would otherwise first queue for LDS, then convert, and only then give
// the matrix cores work (FP32, 27,000 x 96: 0.79 ms against 0.82 before the
// vector adds below, 0.84 with them).
//
// FP64 sums run in NA chains (by u2) that are added at the end: one chain over
// a part of l would add up 16,000 roundings at n = 64,000 in a single part,
// more than the split product of fewer rows and more parts before it did.
template <typename T, int JT> constexpr int ring_chains() {
    return sizeof(T) == 8 ? (JT <= 3 ? 4 : 2) : 1;
}
template <int JT>
__device__ __forceinline__ void ring_products(const RingH<double> &cur, RingH<double> &next,
                                              const unsigned char *hnext, const unsigned char *xb,
                                              int wave, int lane, int64_t,
                                              dv4 (&acc)[1][ring_chains<double, JT>() * JT]) {
    constexpr int NA = ring_chains<double, JT>();
    typedef double v2 __attribute__((ext_vector_type(2)));
    const unsigned xa = lds_addr(xb) + lane * 16;
#pragma unroll
    for (int jt = 0; jt < JT; ++jt) {
        v4f_t x[4];
        const unsigned a = xa + jt * 4096;
        lds_read4(a, a + 1024, a + 2048, a + 3072, x[0], x[1], x[2], x[3]);
#pragma unroll
        for (int u2 = 0; u2 < 4; ++u2) {
            const v2 hv = __builtin_bit_cast(v2, cur.raw[u2]), xv = __builtin_bit_cast(v2, x[u2]);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                dv4 &a4 = acc[0][u2 % NA * JT + jt];
                a4 = __builtin_amdgcn_mfma_f64_16x16x4f64(xv[u], hv[u], a4, 0, 0, 0);
            }
        }
    }
    next.read(hnext, wave, lane);
}

template <int JT>
__device__ __forceinline__ void ring_products(const RingH<float> &cur, RingH<float> &next,
                                              const unsigned char *hnext, const unsigned char *xb,
                                              int wave, int lane, int64_t st, fv4 (&acc)[2][JT]) {
    const unsigned xa = lds_addr(xb) + lane * 16;
    v4f_t xr[2][3];
    lds_read3<1024, 2048>(xa, xr[0][0], xr[0][1], xr[0][2]);
    next.read(hnext, wave, lane);
    // The stage's sums start from zero and are added to the running ones by
    // vector instructions, which round to nearest, with the signs that the
    // fragments carry.
    const float even = __builtin_bit_cast(float, stage_flip(st) ^ 0x3f800000u);
    auto add = [&](fv4 &c, const fv4 &s) {  // element v holds state 4 q + v of the tile
#pragma unroll
        for (int v = 0; v < 4; ++v) c[v] = __builtin_fmaf(v & 1 ? -even : even, s[v], c[v]);
    };
    fv4 sum[2][2];
#pragma unroll
    for (int jt = 0; jt < JT; ++jt) {
        __builtin_amdgcn_sched_barrier(0);
        if (jt + 1 < JT) {
            v4f_t(&x)[3] = xr[(jt + 1) & 1];
            lds_read3<1024, 2048>(xa + (jt + 1) * 3072, x[0], x[1], x[2]);
        }
        const bfv8 x0 = __builtin_bit_cast(bfv8, xr[jt & 1][0]),
                   x1 = __builtin_bit_cast(bfv8, xr[jt & 1][1]),
                   x2 = __builtin_bit_cast(bfv8, xr[jt & 1][2]);
        fv4(&s)[2] = sum[jt & 1];
        s[0] = s[1] = fv4{0, 0, 0, 0};
#define RING_MMA(XV, HV)                                                                    \
    for (int rt = 0; rt < 2; ++rt)                                                          \
        s[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(                                    \
            XV, __builtin_bit_cast(bfv8, cur.HV[rt]), s[rt], 0, 0, 0);
        // smallest terms first
        RING_MMA(x2, h0)
        RING_MMA(x0, h2)
        RING_MMA(x1, h1)
        RING_MMA(x1, h0)
        RING_MMA(x0, h1)
        RING_MMA(x0, h0)
#undef RING_MMA
        if (jt > 0)
            for (int rt = 0; rt < 2; ++rt) add(acc[rt][jt - 1], sum[(jt - 1) & 1][rt]);
        next.split(8 * jt / JT, 8 * (jt + 1) / JT);
        // one product, then three vector instructions of the adds and the
        // split, in turn
#pragma unroll
        for (int i = 0; i < 12; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    for (int rt = 0; rt < 2; ++rt) add(acc[rt][JT - 1], sum[(JT - 1) & 1][rt]);
}

template <typename T, int JT>
__global__ __launch_bounds__(64 * kRingWaves) void dense_ring_kernel(
    int64_t n, int64_t ldh, int32_t k, const T *__restrict__ H, const T *__restrict__ F,
    int32_t ntiles, int32_t nparts, T *__restrict__ P) {
    typedef typename DenseMma<T>::acc_t acc_t;
    constexpr int RT = RingCfg<T>::RT, ROWB = kRingStep * sizeof(T);
    constexpr int XB = JT * RingCfg<T>::PIECES * 1024, HB = ring_rows<T>() * ROWB;
    static_assert(HB == 32768, "each wave loads 4 KB of H per stage");
    constexpr int STAGE = HB + XB;
    constexpr int NB = 3 * STAGE <= 160 * 1024 ? 3 : 2;  // stages in LDS
    constexpr int NQX = (XB / 1024 + kRingWaves - 1) / kRingWaves;
    constexpr int NQ = 4 + NQX;  // loads per wave per stage (a fixed count)
    __shared__ __align__(1024) unsigned char ring[NB * STAGE];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t i0 = (int64_t)blockIdx.x * ring_rows<T>();
    const int part = blockIdx.z;
    const int64_t nst = ldh / kRingStep;
    const int64_t sb = nst * part / nparts, se = nst * (part + 1) / nparts;
    // H: load r of this wave takes 1024 / ROWB rows, one run of ROWB bytes
    // each; the lane at position p of row i takes chunk p ^ (i mod chunks).
    // Rows past n load row n - 1 (never stored).
    constexpr int CPR = ROWB / 16, RPL = 1024 / ROWB;
    int32_t hoff[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 16 * RT * wave + RPL * r + lane / CPR;
        const int64_t last = n - 1 - i0;
        const int64_t ic = i < last ? i : last;
        hoff[r] = (int32_t)(ic * ldh * (int64_t)sizeof(T)) + 16 * ((lane % CPR) ^ (i % CPR));
    }
    const char *hbase = reinterpret_cast<const char *>(H + i0 * ldh);
    const char *fbase = reinterpret_cast<const char *>(F) + (int64_t)blockIdx.y * XB + lane * 16;
    const int64_t fstep = (int64_t)ntiles * RingCfg<T>::PIECES * 1024;
    // stage st to LDS place b; past the last stage: that one again (every
    // wave issues NQ loads a stage)
    auto place = [&](int b) { return ring + b * STAGE; };
    auto fetch_h = [&](int64_t st, int b) {
        unsigned char *d = place(b) + wave * 4096;
        const char *src = hbase + (st < se ? st : se - 1) * ROWB;
#pragma unroll
        for (int r = 0; r < 4; ++r) load_lds_16(src + hoff[r], d + 1024 * r);
    };
    auto fetch_x = [&](int64_t st, int b) {
        unsigned char *d = place(b) + HB;
        const char *src = fbase + (st < se ? st : se - 1) * fstep;
#pragma unroll
        for (int i = 0; i < NQX; ++i) {
            int c = wave + kRingWaves * i;
            c = c < XB / 1024 ? c : XB / 1024 - 1;  // past the last piece: that one again
            load_lds_16(src + 1024 * c, d + 1024 * c);
        }
    };
    constexpr int NA = ring_chains<T, JT>();
    acc_t acc[RT][NA * JT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < NA * JT; ++j) acc[rt][j] = acc_t{0, 0, 0, 0};
    RingH<T> h[2];
    fetch_h(sb, 0);
#pragma unroll
    for (int s = 0; s < NB - 1; ++s) {
        fetch_x(sb + s, s);
        fetch_h(sb + s + 1, s + 1);
    }
    TT_WAIT_VM_LDS((NB - 1) * NQ);  // H of the first stage, this wave's own rows
    h[0].read(place(0), wave, lane);
    h[0].split(0, 8);
    int b = 0;  // place of stage st
    auto step = [&](int64_t st, const RingH<T> &cur, RingH<T> &next) {
        // X of stage st and this wave's H of stage st + 1 are complete when at
        // most the loads of NB - 2 further stages are outstanding; behind the
        // barrier every wave's X is, and every wave has read X of stage
        // st - 1, whose place the next loads take (H of stage st was read
        // during stage st - 1, by the wave that loaded it)
        TT_WAIT_VM_LDS((NB - 2) * NQ);
        line_barrier();
        fetch_x(st + NB - 1, b == 0 ? NB - 1 : b - 1);
        fetch_h(st + NB, b);
        const int bn = b + 1 == NB ? 0 : b + 1;
        ring_products<JT>(cur, next, place(bn), place(b) + HB, wave, lane, st, acc);
        b = bn;
    };
    for (int64_t st = sb; st < se; st += 2) {
        step(st, h[0], h[1]);
        if (st + 1 >= se) break;
        step(st + 1, h[1], h[0]);
    }
    TT_WAIT_ALL();  // no load into LDS may outlive the workgroup
#pragma unroll
    for (int h = NA / 2; h >= 1; h /= 2)  // the chains, pairwise
#pragma unroll
        for (int j = 0; j < h * JT; ++j) acc[0][j] += acc[0][h * JT + j];
    const int li = lane & 15, q = lane >> 4;
    const int c0 = blockIdx.y * 16 * JT;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int64_t r = i0 + 16 * (RT * wave + rt) + li;
        if (r >= n) continue;
        T *Pr = P + ((int64_t)part * n + r) * k;
#pragma unroll
        for (int jt = 0; jt < JT; ++jt)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int c = c0 + 16 * jt + DenseMma<T>::state(q, v);
                if (c < k) Pr[c] = acc[rt][jt][v];
            }
    }
}

// parts of a 32-row tile's list of cnt blocks
__device__ __forceinline__ int block_parts(int64_t cnt, int32_t chunk) {
    return (int)((cnt + chunk - 1) / chunk);
}

// The matrix behind the partial sums as rows, for sums that are not finite: CSR,
// or dense rows of leading dimension ldh (rowptr null).  val null: the partial
// sums stand.
template <typename T> struct RowSource {
    const int64_t *rowptr;
    const int32_t *col;
    const T *val;
    __device__ __forceinline__ double sum(int64_t r, int64_t n, int64_t ldh, const T *x,
                                          int64_t ldx) const {
        const int64_t e0 = rowptr ? rowptr[r] : r * ldh, e1 = rowptr ? rowptr[r + 1] : e0 + n;
        T s = T(0);
        for (int64_t e = e0; e < e1 && s == s; ++e)  // (a NaN stays)
            s += val[e] * x[(rowptr ? (int64_t)col[e] : e - e0) * ldx];
        return (double)s;
    }
};

// One thread per eight rows of one state (the rows of a fragment entry).  With
// blk_ptr the part count is that of the rows' block list (none: no sum).
//
// An infinity or NaN among the states reaches what the rows say: a block's
// zeros times an infinity, or its BF16 pieces, would make NaN of rows without an
// entry there and of infinite results.  Sums that are not finite are therefore
// added up again from the matrix, one entry after the other.
template <typename T>
__global__ __launch_bounds__(256) void dense_combine_kernel(
    int64_t n, int64_t ldh, int32_t k, int32_t nparts, const T *__restrict__ P, const T *X,
    int64_t ldx, const int64_t *__restrict__ ct_rowptr, const int32_t *__restrict__ ct_col,
    const T *__restrict__ ct_val, const T *__restrict__ W, T *Y, int64_t ldy, const T *Z,
    int64_t ldz, double alpha, double beta, double delta, int use_beta, int use_delta,
    int32_t ntiles, T *__restrict__ F, const int64_t *__restrict__ blk_ptr, int32_t chunk,
    RowSource<T> rows) {
    // (fewer than 2^32 threads: k <= 1024, n < 2^25)
    const unsigned e = blockIdx.x * 256u + threadIdx.x;
    const unsigned oc = e / (unsigned)k;
    const int c = (int)(e - oc * (unsigned)k);
    const int64_t o = oc, total = n * k;
    if (o >= ldh / 8) return;
    if (blk_ptr) nparts = block_parts(blk_ptr[(o >> 2) + 1] - blk_ptr[o >> 2], chunk);
    T yv[8], pv[8], xv[8] = {}, zv[8] = {};
    double s[8];
    // (all loads of the eight rows before the first conversion or store)
    auto row = [&](int i) { return 8 * o + i < n ? 8 * o + i : n - 1; };
    if (nparts > 0)
#pragma unroll
        for (int i = 0; i < 8; ++i) pv[i] = P[row(i) * k + c];
    if (use_beta)
#pragma unroll
        for (int i = 0; i < 8; ++i) xv[i] = X[row(i) * ldx + c];
    if (use_delta)
#pragma unroll
        for (int i = 0; i < 8; ++i) zv[i] = Z[row(i) * ldz + c];
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = nparts > 0 ? (double)pv[i] : 0.0;
    // four parts' loads at a time (a small matrix has up to 16 parts: their
    // latency, one after the other, would be most of this kernel)
    for (int p = 1; p < nparts; p += 4) {
        T v[4][8];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int pc = p + u < nparts ? p + u : nparts - 1;
                v[u][i] = P[(int64_t)pc * total + row(i) * k + c];
            }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (p + u < nparts) s[i] += (double)v[u][i];
    }
    if (rows.val) {
        bool finite = true;
#pragma unroll
        for (int i = 0; i < 8; ++i) finite = finite && __builtin_isfinite(s[i]);
        if constexpr (sizeof(T) == 4)
#pragma unroll
            for (int i = 0; i < 8; ++i) s[i] *= 1.0 / kFragScale;
        if (!finite)
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (!__builtin_isfinite(s[i])) s[i] = rows.sum(row(i), n, ldh, X + c, ldx);
    }
    if (ct_rowptr) {
        // entry t of all eight rows together: a row by itself is a serial chain
        // of two loads an entry (12,167 x 37, 19 projectors: 39 -> 30 us)
        int64_t f0[8];
        int len[8], most = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int64_t r = 8 * o + i < n ? 8 * o + i : n - 1;
            f0[i] = ct_rowptr[r];
            len[i] = (int)(ct_rowptr[r + 1] - f0[i]);
            most = len[i] > most ? len[i] : most;
        }
        for (int t = 0; t < most; ++t) {
            double a[8];
            int32_t pr[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {  // (an entry exists: most > 0)
                const int64_t f = t < len[i] ? f0[i] + t : 0;
                a[i] = (double)ct_val[f];
                pr[i] = ct_col[f];
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const double w = (double)W[(int64_t)pr[i] * k + c];
                if (t < len[i]) s[i] += a[i] * w;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int64_t r = 8 * o + i;
        if (r >= n) {
            yv[i] = T(0);
            continue;
        }
        double y = s[i] * alpha;
        if (use_beta) y += beta * (double)xv[i];
        if (use_delta) y += delta * (double)zv[i];
        yv[i] = (T)y;
        Y[r * ldy + c] = yv[i];
    }
    if (F) store_fragment(yv, o, c, ntiles, F);
}

// Block storage of a CSR H_loc: the 32 x 32 blocks that hold an entry, zeros
// included, in the order of their columns, each as operand fragments of its
// two 16-row tiles:
//   FP64: four 1 KB pieces of two doubles per lane, H[row][8 u2 + 2 q + {0, 1}];
//   FP32: two 1 KB pieces of four floats per lane, H[row][8 q + 4 i + 0..3],
// row = lane % 16, q = lane / 16, as the fragments of X have them.
//
// The row kernel above gathers a whole row of X per entry (12,167 x 37, 836
// entries a row: 359 us, bound by those gathers from L2); here an entry costs
// its share of a block (18% full) on the matrix cores.  One wave takes 32 rows' blocks,
// or a part of them, by 16 JT states: H from HBM and X from L2 both come
// straight into registers as whole pieces, no LDS and no barrier, and
// dense_combine_kernel finishes.  A part is at most `chunk` blocks, so that all
// waves have about the same work although rows in the middle of the domain
// have several times the blocks of those at its corners: 141 us, 144 with
// equal part counts.
constexpr int kBlockRows = 32, kBlockElems = 32 * 32;
template <typename T> __device__ __forceinline__ int block_slot(int row, int l);
template <> __device__ __forceinline__ int block_slot<double>(int row, int l) {
    return (row >> 4) * 512 + (l >> 3) * 128 + 2 * ((row & 15) + 16 * ((l >> 1) & 3)) + (l & 1);
}
template <> __device__ __forceinline__ int block_slot<float>(int row, int l) {
    return (row >> 4) * 512 + ((l >> 2) & 1) * 256 + 4 * ((row & 15) + 16 * (l >> 3)) + (l & 3);
}

// Blocks of one 32-row tile per workgroup: bit b of the LDS map is column
// block b.  PASS 0 counts them and notes (count negative) a row whose columns do
// not ascend; PASS 1 lists them and scatters the values.  Duplicate entries add
// up, as in the row kernel: with atomics, in tiles that may hold any.
//
// Bound by latency: a matrix of this size has a few hundred tiles.  Sixteen
// waves take two rows each, and of a run of entries in one block only the first
// sets the map's bit (12,167 rows x 836: count 29 us, FP64 blocks 173, FP32 127;
// 64, 358 and 282 with four waves and atomics for every entry).  With the clear
// and the host's wait for the count an FP64 assembly of that matrix takes 1.61 ms
// in place of 1.25; two products of 37 states (0.19 in place of 0.36 ms each)
// repay that.
constexpr int kBuildThreads = 1024;
template <int PASS, typename T>
__global__ __launch_bounds__(kBuildThreads) void block_build_kernel(
    int64_t n, int32_t words, const int64_t *__restrict__ rowptr, const int32_t *__restrict__ col,
    const T *__restrict__ val, int32_t *__restrict__ count, const int64_t *__restrict__ ptr,
    int32_t *__restrict__ bcol, T *__restrict__ bval) {
    constexpr int NW = kBuildThreads / 64;
    extern __shared__ unsigned block_map[];  // words map words, then their prefix counts
    unsigned *map = block_map, *pre = block_map + words;
    __shared__ int total, disorder;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t tile = blockIdx.x;
    for (int w = t; w < words; w += kBuildThreads) map[w] = 0;
    if (t == 0) total = disorder = 0;
    __syncthreads();
    for (int r = wave; r < kBlockRows; r += NW) {
        const int64_t row = kBlockRows * tile + r;
        if (row >= n) break;
        const int64_t e1 = rowptr[row + 1];
        int last = -1;  // column of the entry before the chunk's first
        for (int64_t base = rowptr[row]; base < e1; base += 64) {
            const bool on = base + lane < e1;
            const int c = on ? col[base + lane] : 0;
            int before = __shfl_up(c, 1);
            if (lane == 0) before = last;
            if (on && (before < 0 || (before >> 5) != (c >> 5)))
                atomicOr(&map[c >> 10], 1u << ((c >> 5) & 31));
            if (PASS == 0 && on && before >= c) disorder = 1;
            last = __shfl(c, 63);
        }
    }
    __syncthreads();
    if (PASS == 0) {
        int c = 0;
        for (int w = t; w < words; w += kBuildThreads) c += __popc(map[w]);
        if (c) atomicAdd(&total, c);
        __syncthreads();
        if (t == 0) count[tile] = disorder ? -total : total;
        return;
    }
    if (wave == 0) {  // prefix counts, 64 words at a time
        int sum = 0;
        for (int w0 = 0; w0 < words; w0 += 64) {
            const int w = w0 + lane, c = w < words ? __popc(map[w]) : 0;
            int s = c;
            for (int o = 1; o < 64; o *= 2) {
                const int x = __shfl_up(s, o);
                if (lane >= o) s += x;
            }
            if (w < words) pre[w] = sum + s - c;
            sum += __shfl(s, 63);
        }
    }
    __syncthreads();
    const int64_t base = ptr[tile];
    for (int w = t; w < words; w += kBuildThreads) {
        unsigned m = map[w];
        for (int64_t b = base + pre[w]; m; ++b) {
            const int bit = __ffs(m) - 1;
            m &= m - 1;
            bcol[b] = 32 * w + bit;
        }
    }
    const bool add = count[tile] < 0;
    for (int r = wave; r < kBlockRows; r += NW) {
        const int64_t row = kBlockRows * tile + r;
        if (row >= n) break;
        for (int64_t e = rowptr[row] + lane; e < rowptr[row + 1]; e += 64) {
            const int c = col[e], w = c >> 10, bit = (c >> 5) & 31;
            const int64_t b = base + pre[w] + __popc(map[w] & ((1u << bit) - 1u));
            T *d = bval + b * kBlockElems + block_slot<T>(r, c & 31);
            if (add)
                atomicAdd(d, val[e]);
            else
                *d = val[e];
        }
    }
}

template <int JT>
__device__ __forceinline__ void block_products(const v4f_t (&h)[2][4], const v4f_t *x, int32_t,
                                               dv4 (&acc)[2][JT]) {
    typedef double v2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int jt = 0; jt < JT; ++jt)
#pragma unroll
        for (int u2 = 0; u2 < 4; ++u2) {
            const v2 xv = __builtin_bit_cast(v2, x[(jt * 4 + u2) * 64]);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                const v2 hv = __builtin_bit_cast(v2, h[rt][u2]);
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    acc[rt][jt] = __builtin_amdgcn_mfma_f64_16x16x4f64(xv[u], hv[u], acc[rt][jt],
                                                                       0, 0, 0);
            }
        }
}
// FP32 as three BF16 pieces, the stage's signs and sums as in the dense product
template <int JT>
__device__ __forceinline__ void block_products(const v4f_t (&h)[2][2], const v4f_t *x, int32_t st,
                                               fv4 (&acc)[2][JT]) {
    bfv8 h0[2], h1[2], h2[2];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        uv4 p0, p1, p2;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            unsigned a, b, c;
            split_bf16(h[rt][i >> 1][2 * (i & 1)], h[rt][i >> 1][2 * (i & 1) + 1], a, b, c);
            p0[i] = a;
            p1[i] = b;
            p2[i] = c;
        }
        h0[rt] = __builtin_bit_cast(bfv8, p0);
        h1[rt] = __builtin_bit_cast(bfv8, p1);
        h2[rt] = __builtin_bit_cast(bfv8, p2);
    }
    const float even = __builtin_bit_cast(float, stage_flip(st) ^ 0x3f800000u);
#pragma unroll
    for (int jt = 0; jt < JT; ++jt) {
        const bfv8 x0 = __builtin_bit_cast(bfv8, x[(jt * 3) * 64]),
                   x1 = __builtin_bit_cast(bfv8, x[(jt * 3 + 1) * 64]),
                   x2 = __builtin_bit_cast(bfv8, x[(jt * 3 + 2) * 64]);
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            fv4 s = {0, 0, 0, 0};
            s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x2, h0[rt], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x0, h2[rt], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x1, h1[rt], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x1, h0[rt], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x0, h1[rt], s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x0, h0[rt], s, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v)
                acc[rt][jt][v] = __builtin_fmaf(v & 1 ? -even : even, s[v], acc[rt][jt][v]);
        }
    }
}

template <typename T, int JT>
__global__ __launch_bounds__(256) void block_spmm_kernel(
    int64_t n, int32_t k, int32_t rtiles, const int64_t *__restrict__ ptr,
    const int32_t *__restrict__ bcol, const T *__restrict__ bval, const T *__restrict__ F,
    int32_t ntiles, int32_t chunk, T *__restrict__ P) {
    typedef typename DenseMma<T>::acc_t acc_t;
    constexpr int HP = sizeof(T) == 8 ? 4 : 2;  // 1 KB pieces of 16 rows of a block
    const int lane = threadIdx.x & 63;
    const int tile = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (tile >= rtiles) return;
    const int part = blockIdx.z;
    const int64_t p0 = ptr[tile], cnt = ptr[tile + 1] - p0;
    const int nparts = block_parts(cnt, chunk);
    if (part >= nparts) return;
    const int64_t b0 = p0 + cnt * part / nparts, b1 = p0 + cnt * (part + 1) / nparts;
    const v4f_t *hp = reinterpret_cast<const v4f_t *>(bval) + lane;
    const v4f_t *xp = reinterpret_cast<const v4f_t *>(F) +
                      (int64_t)blockIdx.y * JT * RingCfg<T>::PIECES * 64 + lane;
    const int64_t xstep = (int64_t)ntiles * RingCfg<T>::PIECES * 64;
    acc_t acc[2][JT];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int jt = 0; jt < JT; ++jt) acc[rt][jt] = acc_t{0, 0, 0, 0};
    if (b0 < b1) {
        v4f_t h[2][HP];
        auto load = [&](int64_t b, v4f_t (&d)[2][HP]) {
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int i = 0; i < HP; ++i) d[rt][i] = hp[((b * 2 + rt) * HP + i) * 64];
        };
        int32_t st = bcol[b0];
        load(b0, h);
        for (int64_t b = b0; b < b1; ++b) {
            const int64_t bn = b + 1 < b1 ? b + 1 : b;
            v4f_t next[2][HP];
            const int32_t stn = bcol[bn];
            load(bn, next);
            block_products<JT>(h, xp + st * xstep, st, acc);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int i = 0; i < HP; ++i) h[rt][i] = next[rt][i];
            st = stn;
        }
    }
    const int li = lane & 15, q = lane >> 4;
    const int c0 = blockIdx.y * 16 * JT;
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        const int64_t r = kBlockRows * (int64_t)tile + 16 * rt + li;
        if (r >= n) continue;
        T *Pr = P + ((int64_t)part * n + r) * k;
#pragma unroll
        for (int jt = 0; jt < JT; ++jt)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int c = c0 + 16 * jt + DenseMma<T>::state(q, v);
                if (c < k) Pr[c] = acc[rt][jt][v];
            }
    }
}

__global__ __launch_bounds__(256) void dense_padding_kernel(int64_t n, int64_t ld, int64_t count,
                                                            double *__restrict__ D) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= count) return;
    const int64_t w = ld - n, cols = n * w;  // columns n .. ld - 1, then rows n ..
    if (e < cols)
        D[e / w * ld + n + e % w] = 0.0;
    else
        D[n * ld + e - cols] = 0.0;
}

// y = H x on the dense storage (+ C^T w where that is not folded in): one
// wavefront per row, 16 bytes of H a lane; HBM-bound (8 n^2 bytes).
__global__ __launch_bounds__(256) void dense_spmv_kernel(
    int64_t n, int64_t ld, const double *__restrict__ D, const double *__restrict__ x,
    const int64_t *__restrict__ ct_rowptr, const int32_t *__restrict__ ct_col,
    const double *__restrict__ ct_val, const double *__restrict__ w, double *__restrict__ y) {
    typedef double v2 __attribute__((ext_vector_type(2)));
    const int lane = threadIdx.x & 63;
    const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= n) return;
    const double *d = D + row * ld;
    double s = 0.0;
    for (int64_t l = 2 * lane; l < n; l += 128) {  // (a pair past n meets the padding of the row)
        const v2 h = *reinterpret_cast<const v2 *>(d + l);
        s += h[0] * x[l];
        if (l + 1 < n) s += h[1] * x[l + 1];
    }
    if (ct_rowptr)
        for (int64_t e = ct_rowptr[row] + lane; e < ct_rowptr[row + 1]; e += 64)
            s += ct_val[e] * w[ct_col[e]];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) y[row] = s;
}

__global__ __launch_bounds__(256) void dense_to_f32_kernel(const double *__restrict__ s,
                                                           float *__restrict__ d, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        d[i] = (float)s[i];
}

unsigned grid_blocks(int64_t n) {
    int64_t b = (n + 255) / 256;
    return (unsigned)(b > 65536 ? 65536 : (b < 1 ? 1 : b));
}

template <typename T, int NC>
int spmm_dispatch_nc(ttdft_ctx ctx, const ttdft_ham_s *H, const T *X, int64_t ldx, const T *W,
                     T *Y, int64_t ldy, const T *Z, int64_t ldz, int32_t k, double alpha,
                     double beta, double delta, int use_beta, int use_delta,
                     const T *val, const T *ct_val) {
    const dim3 grid((unsigned)((H->n + 3) / 4));
    hipLaunchKernelGGL((spmm_fused_kernel<T, NC>), grid, dim3(256), 0, ctx->stream, H->n,
                       H->rowptr, H->col, val, X, ldx, H->p > 0 ? H->ct_rowptr : nullptr,
                       H->ct_col, ct_val, W, k, Y, ldy, Z, ldz, k, (T)alpha, (T)beta,
                       (T)delta, use_beta, use_delta);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

#define TT_NC_SWITCH(NCVAL, CALL)                                                 \
    switch (NCVAL) {                                                              \
    case 1: return CALL(1);                                                       \
    case 2: return CALL(2);                                                       \
    case 3: return CALL(3);                                                       \
    case 4: return CALL(4);                                                       \
    case 5: return CALL(5);                                                       \
    case 6: return CALL(6);                                                       \
    case 7: return CALL(7);                                                       \
    case 8: return CALL(8);                                                       \
    case 9: return CALL(9);                                                       \
    case 10: return CALL(10);                                                     \
    case 11: return CALL(11);                                                     \
    case 12: return CALL(12);                                                     \
    case 13: return CALL(13);                                                     \
    case 14: return CALL(14);                                                     \
    case 15: return CALL(15);                                                     \
    case 16: return CALL(16);                                                     \
    default: break;                                                               \
    }

}  // namespace

int64_t nl_workspace(const ttdft_ham_s *H, int32_t k) {
    const int ns = nl_splits(H, k);
    return (int64_t)H->p * k * (ns > 1 ? 1 + ns : 1);
}

int launch_nl_project(ttdft_ctx ctx, const ttdft_ham_s *H, const void *X, int64_t ldx,
                      int32_t k, int dtype, void *W) {
    if (H->p == 0) return TTDFT_OK;
    TT_CHECK(k >= 1, TTDFT_EBADARG, "k=%d < 1", k);
    if (dtype == TTDFT_F64) {
        TT_CHECK(H->c_val64, TTDFT_EBADARG, "no FP64 copy of the projectors uploaded");
        return nl_launch<double>(ctx, H, (const double *)X, ldx, k, H->c_val64, (double *)W);
    }
    TT_CHECK(H->c_val32, TTDFT_EBADARG, "no FP32 copy of the projectors uploaded");
    return nl_launch<float>(ctx, H, (const float *)X, ldx, k, H->c_val32, (float *)W);
}

int launch_spmm_fused(ttdft_ctx ctx, const ttdft_ham_s *H, const void *X, int64_t ldx,
                      const void *W, void *Y, int64_t ldy, const void *Z, int64_t ldz,
                      int32_t k, int dtype, double alpha, double beta, double delta,
                      int use_beta, int use_delta) {
    const int nc = (k + 63) / 64;
    TT_CHECK(nc >= 1 && nc <= 16, TTDFT_EBADARG, "k=%d outside 1..1024", k);
    if (dtype == TTDFT_F64) {
        TT_CHECK(H->val64, TTDFT_EBADARG, "no FP64 copy of H_loc uploaded");
#define CALL(NCV)                                                                        \
    spmm_dispatch_nc<double, NCV>(ctx, H, (const double *)X, ldx, (const double *)W,     \
                                  (double *)Y, ldy, (const double *)Z, ldz, k, alpha,    \
                                  beta, delta, use_beta, use_delta, H->val64, H->ct_val64)
        TT_NC_SWITCH(nc, CALL)
#undef CALL
    } else {
        TT_CHECK(H->val32, TTDFT_EBADARG, "no FP32 copy of H_loc uploaded");
#define CALL(NCV)                                                                        \
    spmm_dispatch_nc<float, NCV>(ctx, H, (const float *)X, ldx, (const float *)W,        \
                                 (float *)Y, ldy, (const float *)Z, ldz, k, alpha, beta, \
                                 delta, use_beta, use_delta, H->val32, H->ct_val32)
        TT_NC_SWITCH(nc, CALL)
#undef CALL
    }
    return TTDFT_EBADARG;
}

int ham_spmv(ttdft_ctx ctx, const ttdft_ham_s *H, const double *x, double *y) {
    const bool dense = H->format == 2 && H->dense64;
    TT_CHECK(dense || H->val64, TTDFT_EBADARG, "no FP64 copy of H_loc uploaded");
    const bool folded = dense && H->dense_nl;
    double *W = nullptr;
    if (H->p > 0 && !folded) {
        TT_TRY(ctx->scratch[3].ensure((size_t)nl_workspace(H, 1) * sizeof(double)));
        W = (double *)ctx->scratch[3].ptr;
        TT_TRY(launch_nl_project(ctx, H, x, 1, 1, TTDFT_F64, W));
    }
    const int64_t *ctr = H->p > 0 && !folded ? H->ct_rowptr : nullptr;
    const dim3 grid((unsigned)((H->n + 3) / 4));
    if (dense)
        hipLaunchKernelGGL(dense_spmv_kernel, grid, dim3(256), 0, ctx->stream, H->n, H->dense_ld,
                           H->dense64, x, ctr, H->ct_col, H->ct_val64, W, y);
    else
        hipLaunchKernelGGL(spmv_kernel, grid, dim3(256), 0, ctx->stream, H->n, H->rowptr, H->col,
                           H->val64, x, ctr, H->ct_col, H->ct_val64, W, y);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

void drop_dense(ttdft_ham_s *H) {
    dev_release(H->ctx, H->dense64);
    dev_release(H->ctx, H->dense32);
    H->dense64 = nullptr;
    H->dense32 = nullptr;
    H->dense_nl = false;
    if (H->format == 2) H->format = 0;
}

// Dense storage when H_loc has no Kronecker band storage, at least a fifth of
// its entries are nonzero and the FP64 matrix takes at most 48 GiB (n up to
// about 80,000): the CSR kernel then walks rows of thousands of entries with
// the block's k states on one wavefront, while a matrix product streams the
// n^2 values once at full bandwidth.
constexpr double kDenseMaxBytes = 48.0 * 1024 * 1024 * 1024;
bool dense_storage_fits(int64_t n, int64_t nnz) {
    return n >= 1 && 8.0 * (double)n * (double)n <= kDenseMaxBytes &&
           (double)nnz >= 0.2 * (double)n * (double)n;
}
// rows padded to 16 and the leading dimension to 32 (the product's tiles)
int64_t dense_leading_dim(int64_t n) { return (n + 31) / 32 * 32; }
size_t dense_elements(int64_t n) {
    return (size_t)((n + 15) / 16 * 16) * (size_t)dense_leading_dim(n);
}
int launch_dense_padding(ttdft_ctx ctx, int64_t n, double *D) {
    const int64_t ld = dense_leading_dim(n), rows = (n + 15) / 16 * 16;
    const int64_t pad = n * (ld - n) + (rows - n) * ld;
    if (pad == 0) return TTDFT_OK;
    hipLaunchKernelGGL(dense_padding_kernel, dim3((unsigned)((pad + 255) / 256)), dim3(256), 0,
                       ctx->stream, n, ld, pad, D);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}
int maybe_build_dense(ttdft_ctx ctx, ttdft_ham_s *H, int copies) {
    (void)copies;
    const int64_t n = H->n;
    if (H->format != 0 || !dense_storage_fits(n, H->nnz)) return TTDFT_OK;
    const int64_t ld = dense_leading_dim(n);
    const size_t n2 = dense_elements(n);
    const unsigned rows = (unsigned)((n + 3) / 4);
    if (H->val64) {
        TT_TRY(dev_alloc(ctx, (void **)&H->dense64, sizeof(double) * n2));
        TT_HIP(hipMemsetAsync(H->dense64, 0, sizeof(double) * n2, ctx->stream));
        hipLaunchKernelGGL(csr_to_dense_kernel<double>, dim3(rows), dim3(256), 0, ctx->stream, n,
                           ld, H->rowptr, H->col, H->val64, H->dense64);
        TT_LAUNCH_CHECK();
    } else if (H->val32) {
        TT_TRY(dev_alloc(ctx, (void **)&H->dense32, sizeof(float) * n2));
        TT_HIP(hipMemsetAsync(H->dense32, 0, sizeof(float) * n2, ctx->stream));
        hipLaunchKernelGGL(csr_to_dense_kernel<float>, dim3(rows), dim3(256), 0, ctx->stream, n,
                           ld, H->rowptr, H->col, H->val32, H->dense32);
        TT_LAUNCH_CHECK();
    } else {
        return TTDFT_OK;
    }
    H->dense_ld = ld;
    H->dense_nl = false;
    H->format = 2;
    return TTDFT_OK;
}

// Completes the dense storage once the projectors are on the device: the
// nonlocal term C^T D C is added into the FP64 matrix (one rank-p product,
// D C from c_val64 and C from the transposed rows ct_val64), so a product
// with the dense H needs no projection pass; then the FP32 copy is rounded
// from it and the FP64 copy dropped if only FP32 was asked for.  An FP32-only
// build (no FP64 values) keeps the projection pass.
int finish_dense(ttdft_ctx ctx, ttdft_ham_s *H, int copies) {
    if (H->format != 2 || !H->dense64) return TTDFT_OK;
    const int64_t n = H->n, ld = H->dense_ld;
    const size_t n2 = dense_elements(n);
    if (H->p > 0 && H->c_val64 && H->ct_val64) {
        const int64_t p = H->p;
        double *A1 = nullptr, *A2 = nullptr;  // D C as p x n rows, C^T as n x p rows
        TT_TRY(dev_alloc(ctx, (void **)&A1, sizeof(double) * 2 * (size_t)p * n));
        A2 = A1 + p * n;
        int rc = TTDFT_OK;
        hipError_t e = hipMemsetAsync(A1, 0, sizeof(double) * 2 * (size_t)p * n, ctx->stream);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(csr_to_dense_kernel<double>, dim3((unsigned)((p + 3) / 4)),
                               dim3(256), 0, ctx->stream, p, n, H->c_rowptr, H->c_col,
                               H->c_val64, A1);
            hipLaunchKernelGGL(csr_to_dense_kernel<double>, dim3((unsigned)((n + 3) / 4)),
                               dim3(256), 0, ctx->stream, n, p, H->ct_rowptr, H->ct_col,
                               H->ct_val64, A2);
            e = hipGetLastError();
        }
        if (e != hipSuccess) {
            set_error("finish_dense: %s", hipGetErrorString(e));
            rc = TTDFT_EHIP;
        } else {
            // column-major view: H(l, i) = dense[i ld + l] += sum_r (D C)(r, l) C(r, i)
            const double one = 1.0;
            const rocblas_status st = rocblas_dgemm(
                ctx->blas, rocblas_operation_none, rocblas_operation_none, (rocblas_int)n,
                (rocblas_int)n, (rocblas_int)p, &one, A1, (rocblas_int)n, A2, (rocblas_int)p,
                &one, H->dense64, (rocblas_int)ld);
            if (st != rocblas_status_success) {
                set_error("finish_dense: rocblas_dgemm status %d", (int)st);
                rc = TTDFT_ELIB;
            }
        }
        dev_release(ctx, A1);  // reused in stream order
        if (rc != TTDFT_OK) return rc;
        H->dense_nl = true;
    }
    if (copies & TTDFT_HAM_F32) {
        TT_TRY(dev_alloc(ctx, (void **)&H->dense32, sizeof(float) * n2));
        hipLaunchKernelGGL(dense_to_f32_kernel, dim3(grid_blocks((int64_t)n2)), dim3(256), 0,
                           ctx->stream, H->dense64, H->dense32, (int64_t)n2);
        TT_LAUNCH_CHECK();
    }
    if (!(copies & TTDFT_HAM_F64)) {
        dev_release(ctx, H->dense64);
        H->dense64 = nullptr;
    }
    return TTDFT_OK;
}

constexpr int kDenseParts = 16;  // most parts of the split dense and the block product

// 0: one-kernel dense product; 1: form and parts picked; 2..16 and -1..-16:
// split product with that many parts
static int dense_split_form() {
    const char *env = std::getenv("TTDFT_DENSE_LDS");
    return env ? std::atoi(env) : 1;
}

// Tiling of the dense product of k states: fewest columns of at most 96
// states, then the fewest 16-state tiles that cover k in that many columns
// (each column streams H once).
struct DenseTiling {
    int ncol, jt, nparts, chunk = 0;  // chunk: most blocks of a part (block product)
    double stages = 0.0;  // cost of the cheapest dense split, in ring stages
    // one part's sums, all parts' (rounded up to 256 bytes), the fragments of X
    // behind them, and the whole
    size_t part_bytes, partial_bytes, fragment_bytes, bytes;
    DenseTiling(const ttdft_ham_s *H, int32_t k, int dtype) {
        ncol = (k + 95) / 96;
        jt = (k + 16 * ncol - 1) / (16 * ncol);
        part_bytes = (size_t)H->n * k * dtype_size(dtype);
        fragment_bytes = (size_t)((H->n + kRingStep - 1) / kRingStep) * ncol * jt * 1024 *
                         (dtype == TTDFT_F64 ? RingCfg<double>::PIECES : RingCfg<float>::PIECES);
        set_parts(1);
    }
    void set_parts(int p) {
        nparts = p;
        partial_bytes = (p * part_bytes + 255) / 256 * 256;
        bytes = partial_bytes + fragment_bytes;
    }
    // most parts that fit `limit` bytes with the fragments (0: none)
    int parts_within(size_t limit) const {
        if (limit < fragment_bytes + 256) return 0;
        return (int)std::min<size_t>((limit - fragment_bytes - 255) / part_bytes, 1 << 20);
    }
};
// (limit: bytes of work space; nparts is 0 where it holds no part)
static DenseTiling dense_tiling(const ttdft_ham_s *H, int32_t k, int dtype,
                                size_t limit = SIZE_MAX) {
    DenseTiling d(H, k, dtype);
    const int rows = dtype == TTDFT_F64 ? ring_rows<double>() : ring_rows<float>();
    const int64_t nst = H->dense_ld / kRingStep, wgs = (H->n + rows - 1) / rows * d.ncol;
    // Parts of l: one workgroup fills a CU (its LDS stages), so parts p take
    // ceil(wgs p / 256) rounds of nst / p stages and about four to fill and
    // drain the ring; a part's sums cost n k / (64 rows) stages of the chip's
    // bandwidth (written and read back).  The cheapest count is taken.  Where
    // the work space holds only dearer ones, the one-kernel form takes over from
    // 1.25 times the cheapest on in FP64, 2.5 times in FP32 (8,000 and 15,625
    // rows, 96 to 180 states: one kernel 1.4-1.6 and 1.9-3.3 times the split,
    // half the parts 1.9 and 1.5 times).
    const int within = d.parts_within(limit);
    const int form = dense_split_form();
    if (form != 1) {
        d.set_parts((int)std::min<int64_t>({std::abs(form), kDenseParts, nst, within}));
        return d;
    }
    double best = 0.0, best_within = 0.0;
    int nparts = 0;
    for (int p = 1; p <= kDenseParts && p <= nst; ++p) {
        const double cost = (double)((wgs * p + 255) / 256) * (double)((nst + p - 1) / p + 4) +
                            p * (double)H->n * k / (256.0 * 16 * rows);
        if (p == 1 || cost < best) best = cost;
        if (p <= within && (p == 1 || cost < best_within)) {
            best_within = cost;
            nparts = p;
        }
    }
    d.set_parts(best_within <= (dtype == TTDFT_F64 ? 1.25 : 2.5) * best ? nparts : 0);
    d.stages = best;
    return d;
}

// Does the dense product of k states run as the split product?  From 8,192 rows
// on (8,000 x 24 FP64 1,344 us in one kernel, 953 split, a filter of nine
// products; 8,000 x 1 FP32 391 / 488).  Below, the cheaper of two costs in us, by
// 16-state tiles and type:  the split's two further launches and its ring
// stages (dense_tiling), against the one kernel's rounds of 256 workgroups of 16
// rows, one a CU, that each walk all of l.  Fitted to filters of 512 to 8,000
// rows with 1 to 400 states, of which it loses 0.3% against the better form.
// One kernel / split, us, FP64: 512 x 16 64 / 131; 1,331 x 200 246 / 339;
// 1,728 x 200 537 / 419; 4,096 x 96 563 / 637; 4,913 x 16 520 / 359.
// FP32: 1,728 x 96 224 / 293, x 300 435 / 337; 2,744 x 80 313 / 302; 4,096 x 24
// 201 / 235, x 96 461 / 393.
static bool dense_split(const ttdft_ham_s *H, int32_t k, int dtype) {
    const int form = dense_split_form();
    if (form != 1) return form != 0;
    if (H->n > 8192) return true;
    static const struct {
        double split, stage, one, row;
    } cost[2][6] = {{{8.2, 1.13, 3.8, 0.0056},
                     {9.3, 1.31, 4.6, 0.0078},
                     {8.2, 1.74, 6.1, 0.0103},
                     {7.2, 2.11, 7.0, 0.0135},
                     {2.9, 2.66, 7.1, 0.0146},
                     {4.0, 2.67, 5.7, 0.0162}},
                    {{6.5, 1.25, 3.8, 0.0024},
                     {8.2, 1.20, 3.6, 0.0048},
                     {8.6, 1.40, 4.4, 0.0067},
                     {11.5, 1.49, 4.4, 0.0098},
                     {12.3, 1.70, 4.4, 0.0118},
                     {12.7, 1.87, 3.7, 0.0135}}};
    const DenseTiling d = dense_tiling(H, k, dtype);
    const auto &c = cost[dtype == TTDFT_F64 ? 0 : 1][d.jt - 1];
    const int64_t rounds = ((H->n + 15) / 16 * d.ncol + 255) / 256;
    return c.split + c.stage * d.stages < c.one + c.row * (double)(rounds * H->dense_ld);
}

template <typename T, int JT>
static void dense_launch(ttdft_ctx ctx, const ttdft_ham_s *H, const T *Hd, const T *ctv,
                         const void *X, int64_t ldx, const void *W, void *Y, int64_t ldy,
                         const void *Z, int64_t ldz, int32_t k, double alpha, double beta,
                         double delta, int use_beta, int use_delta, const DenseTiling &d, void *P,
                         StepChain chain) {
    const int64_t n = H->n;
    const dim3 grid((unsigned)((n + 15) / 16), (unsigned)((k + 16 * JT - 1) / (16 * JT)));
    const int64_t *ctr = H->p > 0 && !H->dense_nl ? H->ct_rowptr : nullptr;
    // Split product against the one-kernel form, which is for small matrices
    // and callers whose work space cannot hold the partial sums: FP32
    // 27,000 x 96 0.84 + 0.03 (sum of the parts) against 2.54 ms, FP64
    // 8,000 x 24 0.108 + 0.007 against 0.153.  TTDFT_DENSE_LDS=0 turns the split
    // off, 1 picks the form and the parts, 2..16 and -1..-16 split into that many.
    if (P) {
        const int ntiles = d.ncol * JT;
        T *Pt = (T *)P, *F = (T *)((char *)P + d.partial_bytes);
        const unsigned cb = (unsigned)((H->dense_ld / 8 * k + 255) / 256);
        if (!chain.have)
            hipLaunchKernelGGL((x_fragments_kernel<T>), dim3(cb), dim3(256), 0, ctx->stream, n,
                               H->dense_ld, k, (const T *)X, ldx, ntiles, F);
        const dim3 g((unsigned)((n + ring_rows<T>() - 1) / ring_rows<T>()), (unsigned)d.ncol,
                     (unsigned)d.nparts);
        hipLaunchKernelGGL((dense_ring_kernel<T, JT>), g, dim3(64 * kRingWaves), 0,
                           ctx->stream, n, H->dense_ld, k, Hd, F, ntiles, d.nparts, Pt);
        hipLaunchKernelGGL((dense_combine_kernel<T>), dim3(cb), dim3(256), 0, ctx->stream, n,
                           H->dense_ld, k, d.nparts, Pt, (const T *)X, ldx, ctr, H->ct_col, ctv,
                           (const T *)W, (T *)Y, ldy, (const T *)Z, ldz, alpha, beta, delta,
                           use_beta, use_delta, ntiles, chain.want ? F : nullptr, nullptr, 0,
                           RowSource<T>{nullptr, nullptr, sizeof(T) == 4 ? Hd : nullptr});
        return;
    }
    // six-state runs per lane, fetched as pairs, when every tile is full and
    // every row of X starts on a pair boundary (even leading dimension and a
    // pair-aligned X: a filter block may start at an odd column)
    if (JT == 6 && k % (16 * JT) == 0 && ldx % 2 == 0 &&
        reinterpret_cast<uintptr_t>(X) % (2 * sizeof(T)) == 0)
        hipLaunchKernelGGL((dense_hx_kernel<T, JT, (JT == 6)>), grid, dim3(64 * kDenseWaves), 0,
                           ctx->stream, n, H->dense_ld, k, Hd, (const T *)X, ldx, ctr, H->ct_col,
                           ctv, (const T *)W, (T *)Y, ldy, (const T *)Z, ldz, alpha, beta, delta,
                           use_beta, use_delta);
    else
        hipLaunchKernelGGL((dense_hx_kernel<T, JT, false>), grid, dim3(64 * kDenseWaves), 0,
                           ctx->stream, n, H->dense_ld, k, Hd, (const T *)X, ldx, ctr, H->ct_col,
                           ctv, (const T *)W, (T *)Y, ldy, (const T *)Z, ldz, alpha, beta, delta,
                           use_beta, use_delta);
}

// H X on the dense storage with the recurrence epilogue in one kernel; the
// state tiles per workgroup follow k (16 to 96 states)
static int launch_dense_spmm(ttdft_ctx ctx, const ttdft_ham_s *H, const void *X, int64_t ldx,
                             const void *W, void *Y, int64_t ldy, const void *Z, int64_t ldz,
                             int32_t k, int dtype, double alpha, double beta, double delta,
                             int use_beta, int use_delta, const DenseTiling &d, void *P,
                             StepChain chain) {
#define DENSE_CASE(JTV)                                                                         \
    case JTV:                                                                                   \
        if (dtype == TTDFT_F64)                                                                 \
            dense_launch<double, JTV>(ctx, H, H->dense64, H->ct_val64, X, ldx, W, Y, ldy, Z,    \
                                      ldz, k, alpha, beta, delta, use_beta, use_delta, d, P,    \
                                      chain);                                                   \
        else                                                                                    \
            dense_launch<float, JTV>(ctx, H, H->dense32, H->ct_val32, X, ldx, W, Y, ldy, Z,     \
                                     ldz, k, alpha, beta, delta, use_beta, use_delta, d, P,     \
                                     chain);                                                    \
        break;
    switch (d.jt) {
        DENSE_CASE(1)
        DENSE_CASE(2)
        DENSE_CASE(3)
        DENSE_CASE(4)
        DENSE_CASE(5)
        DENSE_CASE(6)
    default:
        break;
    }
#undef DENSE_CASE
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

void drop_blocks(ttdft_ham_s *H) {
    dev_release(H->ctx, H->blk_ptr);
    dev_release(H->ctx, H->blk_col);
    dev_release(H->ctx, H->blk64);
    dev_release(H->ctx, H->blk32);
    dev_release(H->ctx, H->blk_count);
    H->blk_count = nullptr;
    H->blk_ptr = nullptr;
    H->blk_col = nullptr;
    H->blk64 = nullptr;
    H->blk32 = nullptr;
    H->nblk = 0;
}

// Blocks of a CSR H_loc when they are full enough: from 10% of their places on,
// where the products of most state counts gain (block_product_pays) and the
// storage (8 bytes a place against 12 an entry) is at most 7 times that of the
// rows.  Only the precisions asked for are built: a device assembly still holds
// its FP64 rows here when FP32 alone was.
static int try_build_blocks(ttdft_ctx ctx, ttdft_ham_s *H, int copies) {
    const int64_t n = H->n;
    const int64_t words = (n + 1023) / 1024, tiles = (n + kBlockRows - 1) / kBlockRows;
    const bool f64 = H->val64 && (copies & TTDFT_HAM_F64);
    const bool f32 = H->val32 && (copies & TTDFT_HAM_F32);
    if (H->format != 0 || (!f64 && !f32) || H->nnz < 1 || words > 4096) return TTDFT_OK;
    TT_TRY(dev_alloc(ctx, (void **)&H->blk_count, sizeof(int32_t) * tiles));
    const size_t lds = sizeof(unsigned) * 2 * (size_t)words;
    const dim3 grid((unsigned)tiles), block(kBuildThreads);
    hipLaunchKernelGGL((block_build_kernel<0, double>), grid, block, lds, ctx->stream, n,
                       (int32_t)words, H->rowptr, H->col, nullptr, H->blk_count, nullptr, nullptr,
                       nullptr);
    TT_LAUNCH_CHECK();
    std::vector<int32_t> cnt(tiles);
    TT_HIP(hipMemcpyAsync(cnt.data(), H->blk_count, sizeof(int32_t) * tiles,
                          hipMemcpyDeviceToHost, ctx->stream));
    TT_HIP(hipStreamSynchronize(ctx->stream));
    std::vector<int64_t> &ptr = H->blk_ptr_host;  // (read by the copy below after the return)
    ptr.assign(tiles + 1, 0);
    for (int64_t t = 0; t < tiles; ++t) {
        const int64_t c = std::abs(cnt[t]);
        ptr[t + 1] = ptr[t] + c;
        H->blk_most = std::max(H->blk_most, c);
    }
    const int64_t nblk = ptr[tiles];
    if ((double)H->nnz < 0.1 * kBlockElems * (double)nblk ||
        8.0 * kBlockElems * (double)nblk > kDenseMaxBytes) {
        drop_blocks(H);
        return TTDFT_OK;
    }
    H->nblk = nblk;
    TT_TRY(dev_alloc(ctx, (void **)&H->blk_ptr, sizeof(int64_t) * (tiles + 1)));
    TT_TRY(dev_alloc(ctx, (void **)&H->blk_col, sizeof(int32_t) * nblk));
    TT_HIP(hipMemcpyAsync(H->blk_ptr, ptr.data(), sizeof(int64_t) * (tiles + 1),
                          hipMemcpyHostToDevice, ctx->stream));
    if (f64) {
        TT_TRY(dev_alloc(ctx, (void **)&H->blk64, sizeof(double) * kBlockElems * nblk));
        TT_HIP(hipMemsetAsync(H->blk64, 0, sizeof(double) * kBlockElems * nblk, ctx->stream));
        hipLaunchKernelGGL((block_build_kernel<1, double>), grid, block, lds, ctx->stream, n,
                           (int32_t)words, H->rowptr, H->col, H->val64, H->blk_count, H->blk_ptr,
                           H->blk_col, H->blk64);
    }
    if (f32) {
        TT_TRY(dev_alloc(ctx, (void **)&H->blk32, sizeof(float) * kBlockElems * nblk));
        TT_HIP(hipMemsetAsync(H->blk32, 0, sizeof(float) * kBlockElems * nblk, ctx->stream));
        hipLaunchKernelGGL((block_build_kernel<1, float>), grid, block, lds, ctx->stream, n,
                           (int32_t)words, H->rowptr, H->col, H->val32, H->blk_count, H->blk_ptr,
                           H->blk_col, H->blk32);
    }
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

// The rows are whole without the blocks: where these find no memory, the row
// kernel takes every product.
int build_blocks(ttdft_ctx ctx, ttdft_ham_s *H, int copies) {
    const int rc = try_build_blocks(ctx, H, copies);
    if (rc != TTDFT_OK) drop_blocks(H);
    if (rc != TTDFT_ENOMEM) return rc;
    clear_error();
    return TTDFT_OK;
}

// Does a product of k states run by blocks?  Both forms' times go with what they
// read: the row kernel's with its entries, once per 64 states (FP64 33 ps each
// time, FP32 12 ps and 9 ps each time), the block kernel's with its blocks, once
// per column of at most 96 states, and their 16-state tiles (1.6 ns and 0.55 ns a
// tile in FP64, 0.8 and 0.31 in FP32).  Measured, rows / blocks in us:
//   15,625 rows, blocks 10% full: FP64 16 states 203 / 147, 64 207 / 225, 96
//   385 / 347; FP32 16 147 / 83, 64 148 / 134, 128 179 / 230;
//   21,952 rows, 16% full: FP64 64 609 / 401, 300 3,902 / 1,891; FP32 64
//   426 / 243, 300 1,075 / 1,136;
//   12,167 rows, 18% full: FP64 16 364 / 150, 300 1,806 / 854; FP32 16
//   265 / 81, 300 701 / 463.
// TTDFT_CSR_BLOCKS=0 takes the rows, 1 the blocks wherever they are stored.
static bool block_product_pays(const ttdft_ham_s *H, int32_t k, int dtype) {
    if (const char *env = std::getenv("TTDFT_CSR_BLOCKS")) return std::atoi(env) != 0;
    const DenseTiling d(H, k, dtype);
    const int nc = (k + 63) / 64;
    const bool f64 = dtype == TTDFT_F64;
    const double entry = f64 ? 0.033 * nc : 0.012 + 0.009 * nc;
    const double block = d.ncol * (f64 ? 1.6 + 0.55 * d.jt : 0.8 + 0.31 * d.jt);
    return entry * (double)H->nnz >= block * (double)H->nblk;
}

// State tiles, parts and work space of the block product: chunks of blocks for
// about four waves per SIMD in FP64, two in FP32 (there the partial sums weigh
// more: 12,167 x 64 119 us against 139), four blocks at least, and as long as
// keeps the longest list to kDenseParts parts: every part has a place for all
// rows, so one full row tile in a sparse matrix would otherwise take gigabytes
// (200,000 rows x 64 states with 32 full rows: 91 GB).
static DenseTiling block_tiling(const ttdft_ham_s *H, int32_t k, int dtype,
                                size_t limit = SIZE_MAX) {
    DenseTiling d(H, k, dtype);
    const int64_t most = std::min(kDenseParts, d.parts_within(limit));
    if (most < 1) {
        d.set_parts(0);
        return d;
    }
    const int64_t waves = dtype == TTDFT_F64 ? 4096 : 2048;
    d.chunk = (int)std::max<int64_t>(
        {(H->nblk * d.ncol + waves - 1) / waves, 4, (H->blk_most + most - 1) / most});
    d.set_parts((int)((H->blk_most + d.chunk - 1) / d.chunk));
    return d;
}

template <typename T, int JT>
static void block_launch(ttdft_ctx ctx, const ttdft_ham_s *H, const DenseTiling &d, const T *val,
                         const T *bval, const T *ctv, const void *X, int64_t ldx, const void *W, void *Y,
                         int64_t ldy, const void *Z, int64_t ldz, int32_t k, double alpha,
                         double beta, double delta, int use_beta, int use_delta, void *P,
                         StepChain chain) {
    const int64_t n = H->n, ld = dense_leading_dim(n);
    const int ntiles = d.ncol * JT, rtiles = (int)((n + kBlockRows - 1) / kBlockRows);
    T *Pt = (T *)P, *F = (T *)((char *)P + d.partial_bytes);
    const unsigned cb = (unsigned)((ld / 8 * k + 255) / 256);
    if (!chain.have)
        hipLaunchKernelGGL((x_fragments_kernel<T>), dim3(cb), dim3(256), 0, ctx->stream, n, ld, k,
                           (const T *)X, ldx, ntiles, F);
    const dim3 g((unsigned)((rtiles + 3) / 4), (unsigned)d.ncol, (unsigned)d.nparts);
    hipLaunchKernelGGL((block_spmm_kernel<T, JT>), g, dim3(256), 0, ctx->stream, n, k, rtiles,
                       H->blk_ptr, H->blk_col, bval, F, ntiles, d.chunk, Pt);
    hipLaunchKernelGGL((dense_combine_kernel<T>), dim3(cb), dim3(256), 0, ctx->stream, n, ld, k,
                       d.nparts, Pt, (const T *)X, ldx, H->p > 0 ? H->ct_rowptr : nullptr,
                       H->ct_col, ctv, (const T *)W, (T *)Y, ldy, (const T *)Z, ldz, alpha, beta,
                       delta, use_beta, use_delta, ntiles, chain.want ? F : nullptr, H->blk_ptr,
                       d.chunk, RowSource<T>{H->rowptr, H->col, val});
}

static int launch_block_spmm(ttdft_ctx ctx, const ttdft_ham_s *H, const void *X, int64_t ldx,
                             const void *W, void *Y, int64_t ldy, const void *Z, int64_t ldz,
                             int32_t k, int dtype, double alpha, double beta, double delta,
                             int use_beta, int use_delta, const DenseTiling &d, void *P,
                             StepChain chain) {
#define BLOCK_CASE(JTV)                                                                        \
    case JTV:                                                                                  \
        if (dtype == TTDFT_F64)                                                                \
            block_launch<double, JTV>(ctx, H, d, H->val64, H->blk64, H->ct_val64, X, ldx, W, Y, \
                                      ldy, Z, ldz, k, alpha, beta, delta, use_beta, use_delta, P,      \
                                      chain);                                                  \
        else                                                                                   \
            block_launch<float, JTV>(ctx, H, d, H->val32, H->blk32, H->ct_val32, X, ldx, W, Y,  \
                                     ldy, Z, ldz, k, alpha, beta, delta, use_beta, use_delta, P,       \
                                     chain);                                                   \
        break;
    switch (d.jt) {
        BLOCK_CASE(1)
        BLOCK_CASE(2)
        BLOCK_CASE(3)
        BLOCK_CASE(4)
        BLOCK_CASE(5)
        BLOCK_CASE(6)
    default:
        break;
    }
#undef BLOCK_CASE
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int ham_step(ttdft_ctx ctx, const ttdft_ham_s *H, const void *X, int64_t ldx, void *Y,
             int64_t ldy, const void *Z, int64_t ldz, int32_t k, int dtype, double alpha,
             double beta, double delta, int use_beta, int use_delta, void *ws,
             size_t ws_bytes, StepChain *chain) {
    const size_t es = dtype_size(dtype);
    const bool band = H->format == 1 && k >= 16 &&
                      (dtype == TTDFT_F64 ? H->mf64 != nullptr : H->mf32 != nullptr);
    const bool dense = H->format == 2 && (dtype == TTDFT_F64 ? H->dense64 != nullptr
                                                            : H->dense32 != nullptr);
    // (from 8 states on: below, a block's columns are mostly padding)
    const bool blocks = H->format == 0 && k >= 8 && k <= 1024 &&
                        (dtype == TTDFT_F64 ? H->blk64 != nullptr : H->blk32 != nullptr) &&
                        block_product_pays(H, k, dtype);
    void *W = nullptr;
    if (H->p > 0 && !(dense && H->dense_nl)) {  // folded into the dense storage otherwise
        const size_t need = (size_t)nl_workspace(H, k) * es;
        if (ws) {
            TT_CHECK(need <= ws_bytes, TTDFT_EBADARG,
                     "the nonlocal projection of %d projectors x %d states needs %zu bytes of "
                     "work space, more than the %zu available",
                     H->p, k, need, ws_bytes);
            W = ws;
        } else {
            TT_TRY(ctx->scratch[3].ensure(need));
            W = ctx->scratch[3].ptr;
        }
        PendingTiming tn;
        TT_TRY(timing_begin(ctx, TTDFT_KSTAT_NLPROJ, &tn));
        TT_TRY(launch_nl_project(ctx, H, X, ldx, k, dtype, W));
        TT_TRY(timing_end(ctx, &tn, (double)H->nnz_c * (es + 4) + (double)H->nnz_c * k * es,
                          2.0 * H->nnz_c * k));
    }
    PendingTiming ts;
    TT_TRY(timing_begin(ctx, TTDFT_KSTAT_SPMM, &ts));
    if (band)
        TT_TRY(launch_band_spmm(ctx, H, X, ldx, W, Y, ldy, Z ? Z : Y, Z ? ldz : ldy, k, dtype,
                                alpha, beta, delta, use_beta, use_delta));
    else {
        // Partial sums and fragments of the split dense and the block product:
        // after the projections in the caller's work space, in as many parts as
        // that holds, else from the context.  Where the caller's work space
        // holds no part, or the context finds no memory, the product runs in one
        // kernel.  (The same result up to the order of the additions.)
        void *P = nullptr;
        DenseTiling tiling(H, k, dtype);
        if (blocks || (dense && dense_split(H, k, dtype))) {
            const size_t off = W ? ((size_t)nl_workspace(H, k) * es + 255) / 256 * 256 : 0;
            const size_t limit = !ws ? SIZE_MAX : off < ws_bytes ? ws_bytes - off : 0;
            tiling = blocks ? block_tiling(H, k, dtype, limit) : dense_tiling(H, k, dtype, limit);
            if (ws) {
                if (tiling.nparts > 0) P = (char *)ws + off;
            } else if (ctx->scratch[8].ensure(tiling.bytes) == TTDFT_OK) {
                P = ctx->scratch[8].ptr;
            } else {
                clear_error();
            }
        }
        StepChain now;  // what this step finds and is to leave
        if (chain && P) now = *chain;
        if (chain) chain->have = P && chain->want;
        const void *Zp = Z ? Z : Y;
        const int64_t ldzp = Z ? ldz : ldy;
        if (dense)
            TT_TRY(launch_dense_spmm(ctx, H, X, ldx, W, Y, ldy, Zp, ldzp, k, dtype, alpha, beta,
                                     delta, use_beta, use_delta, tiling, P, now));
        else if (blocks && P)
            TT_TRY(launch_block_spmm(ctx, H, X, ldx, W, Y, ldy, Zp, ldzp, k, dtype, alpha, beta,
                                     delta, use_beta, use_delta, tiling, P, now));
        else
            TT_TRY(launch_spmm_fused(ctx, H, X, ldx, W, Y, ldy, Zp, ldzp, k, dtype, alpha, beta,
                                     delta, use_beta, use_delta));
    }
    // algorithmic bytes: H_loc values + indices + row pointers, X panel read once,
    // Y written once, the recurrence operands read once (fused epilogue).
    const double nk = (double)H->n * k * es;
    const double bytes = (double)H->nnz * (es + 4) + 8.0 * (H->n + 1) + nk + nk +
                         (use_delta ? nk : 0.0);
    const double flops = 2.0 * H->nnz * k + 5.0 * H->n * k;
    TT_TRY(timing_end(ctx, &ts, bytes, flops));
    return TTDFT_OK;
}

}  // namespace ttdft
