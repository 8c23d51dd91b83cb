// Layers of the 3-D convolutional network that predicts a correction to the
// atomic-superposition initial density (dft/InitialGuess.cc:573-762 is the
// start it corrects; the network has no reference counterpart).
//
// Tensors are one sample's [C][D][H][W] FP32 arrays (x fastest); a channel
// concatenation is two adjacent channel blocks, so it costs nothing.
//
// Convolutions (kernel ks = 1 or 3, stride 1, zero padding ks / 2) are implicit
// GEMMs on the matrix cores, in BF16 (operands rounded as they are staged into
// LDS, FP32 accumulation) or FP32.  Tensors and weights stay FP32 in HBM.
//   forward:         Y[co][p] = sum_{c,tap} W[co][c][tap] X[c][p + tap]
//   backward data:   the same with W'[ci][co][ks^3-1-t] = W[co][ci][t]
//   backward weight: dW[co][c][tap] = sum_p dY[co][p] X[c][p + tap], split over
//                    position ranges; the partial sums are added in a fixed order.
#include <algorithm>
#include <cmath>
#include <vector>

#include "internal.h"

namespace ttdft {
namespace {

struct Geo {
    int32_t D, H, W;
    int64_t P;
};

// ---- convolutions on the matrix cores ------------------------------------------
// One MFMA step takes a 16-byte vector of operand elements per lane: eight BF16
// values (one v_mfma_f32_16x16x32_bf16) or four FP32 values (four
// v_mfma_f32_16x16x4_f32, the u-th pairing element u of every lane).  Operand A
// sits in lanes i + 16 g (row i), operand B in lanes j + 16 g (column j); the
// vector of lane group g holds the same inner indices in both.  Element v of
// lane l of the result is D[4 (l/16) + v][l%16].
typedef float f4v __attribute__((ext_vector_type(4)));
typedef short s8v __attribute__((ext_vector_type(8)));
typedef __bf16 b8v __attribute__((ext_vector_type(8)));

struct Bf16Op {
    typedef unsigned short elem;
    typedef s8v vec;
    static constexpr int VE = 8;
    static __device__ __forceinline__ elem cvt(float x) {
        return __builtin_bit_cast(unsigned short, (__bf16)x);  // nearest even
    }
    static __device__ __forceinline__ f4v mma(vec a, vec b, f4v c) {
#if defined(__HIP_DEVICE_COMPILE__)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8v, a),
                                                       __builtin_bit_cast(b8v, b), c, 0, 0, 0);
#else
        return c;
#endif
    }
};
struct F32Op {
    typedef float elem;
    typedef f4v vec;
    static constexpr int VE = 4;
    static __device__ __forceinline__ elem cvt(float x) { return x; }
    static __device__ __forceinline__ f4v mma(vec a, vec b, f4v c) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b[u], c, 0, 0, 0);
        return c;
    }
};

// Weights in operand order: vector ((mt nchunk + chunk) nsteps + step) 64 + lane
// holds output channel 16 mt + lane%16 against the VE input channels
// chunk NG VE + (g%NG) VE .. of tap step (4/NG) + g/NG, g = lane/16 (zero past
// the last channel or tap).  flip: the transposed, mirrored weights of the
// data gradient (m and c exchange roles in the stored W[c][m][tap]).
template <typename OP>
__global__ __launch_bounds__(256) void conv_weights_kernel(const float *__restrict__ W, int M,
                                                           int C, int KT, int flip, int NG,
                                                           int nchunk, int nsteps,
                                                           int64_t total,
                                                           typename OP::elem *__restrict__ out) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= total) return;
    const int lane = (int)(e & 63), g = lane >> 4;
    int r = (int)(e >> 6);
    const int step = r % nsteps;
    r /= nsteps;
    const int chunk = r % nchunk, m = 16 * (r / nchunk) + (lane & 15);
    const int tap = step * (4 / NG) + g / NG, c0 = (chunk * NG + g % NG) * OP::VE;
    typename OP::vec w;
#pragma unroll
    for (int v = 0; v < OP::VE; ++v) {
        const int c = c0 + v;
        float x = 0.0f;
        if (m < M && c < C && tap < KT)
            x = flip ? W[((int64_t)c * M + m) * KT + KT - 1 - tap]
                     : W[((int64_t)m * C + c) * KT + tap];
        w[v] = OP::cvt(x);
    }
    *reinterpret_cast<typename OP::vec *>(out + e * OP::VE) = w;
}

// Y[m][p] (=|+=) b[m] + sum_{c,tap} W[m][c][tap] X[c][p + tap]
// A workgroup owns TX x TY x TZ positions and 16 NM output channels.  Per chunk
// of NG VE input channels it stages the positions and their halo in LDS once,
// channels innermost (one 16-byte vector per position and channel group, the
// position pitch one vector more than NG so that 16 neighbouring positions fall
// on distinct banks), and every tap reads the same stage at its offset: an
// element is loaded and converted once for 27 taps, where a gather per tap
// bounded the kernel before.  4 waves split the positions; a wave's B vectors
// serve its NM row tiles.  What bounds it now is the staging of the halo
// (2.3-2.5 times the positions at 256 positions per workgroup).
// Measured (64^3 network, whole training step): 27 products of a pass 7.8 ms
// before, 0.71 ms now with the weights brought into operand order.
template <typename OP, int KS, int NG, int TX, int TY, int TZ, int NM>
__global__ __launch_bounds__(256) void conv_kernel(const float *__restrict__ X, int ci, Geo g,
                                                   const typename OP::elem *__restrict__ Wf,
                                                   const float *__restrict__ bias, int co,
                                                   float *__restrict__ Y, int accumulate,
                                                   int nchunk, int ntx, int nty) {
    typedef typename OP::elem elem;
    typedef typename OP::vec vec;
    constexpr int VE = OP::VE, KT = KS * KS * KS, PAD = KS / 2;
    constexpr int HX = TX + KS - 1, HY = TY + KS - 1, HZ = TZ + KS - 1, NH = HX * HY * HZ;
    constexpr int PITCH = (NG + 1) * VE;
    constexpr int NS = (KT * NG + 3) / 4;     // MFMA steps per chunk
    constexpr int NP = TX * TY * TZ / 64;     // 16-position tiles per wave
    __shared__ __align__(16) elem xs[NH * PITCH];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int li = lane & 15, lg = lane >> 4;
    const int mt0 = blockIdx.y * NM;
    int b = blockIdx.x;
    const int x0 = (b % ntx) * TX;
    b /= ntx;
    const int y0 = (b % nty) * TY, z0 = (b / nty) * TZ;
    // halo slot of this lane's position in each of its tiles, at its channel group
    int base[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) {
        const int p = (wave * NP + q) * 16 + li;
        base[q] = (((p / (TX * TY)) * HY + (p / TX) % TY) * HX + p % TX) * PITCH + (lg % NG) * VE;
    }
    f4v acc[NM][NP];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int q = 0; q < NP; ++q) acc[m][q] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
    const elem *wl = Wf + lane * VE;
    for (int chunk = 0; chunk < nchunk; ++chunk) {
        const int c0 = chunk * NG * VE;
        if (chunk) __syncthreads();
        for (int e = t; e < NH * NG; e += 256) {
            const int pos = e % NH, cg = e / NH;
            const int x = x0 + pos % HX - PAD, y = y0 + (pos / HX) % HY - PAD,
                      z = z0 + pos / (HX * HY) - PAD;
            const bool in = x >= 0 && x < g.W && y >= 0 && y < g.H && z >= 0 && z < g.D;
            // unconditional loads (element 0 where there is none), so that they
            // are in flight together
            const int64_t o = in ? ((int64_t)z * g.H + y) * g.W + x : 0;
            float f[VE];
#pragma unroll
            for (int v = 0; v < VE; ++v) {
                const int c = c0 + cg * VE + v;
                f[v] = X[c < ci ? (int64_t)c * g.P + o : 0];
            }
            vec w;
#pragma unroll
            for (int v = 0; v < VE; ++v)
                w[v] = OP::cvt(in && c0 + cg * VE + v < ci ? f[v] : 0.0f);
            *reinterpret_cast<vec *>(&xs[pos * PITCH + cg * VE]) = w;
        }
        __syncthreads();
        auto load_w = [&](int s, vec (&w)[NM]) {
#pragma unroll
            for (int m = 0; m < NM; ++m)
                w[m] = *reinterpret_cast<const vec *>(
                    wl + (((int64_t)(mt0 + m) * nchunk + chunk) * NS + s) * 64 * VE);
        };
        vec wa[NM], wb[NM];
        load_w(0, wa);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (s + 1 < NS) load_w(s + 1, wb);
            int off = 0;
            if constexpr (KS == 3) {
                constexpr int TS = 4 / NG;  // taps per step
#pragma unroll
                for (int u = 0; u < TS; ++u) {
                    const int tap = s * TS + u < KT ? s * TS + u : KT - 1;
                    const int o = (((tap / 9) * HY + (tap / 3) % 3) * HX + tap % 3) * PITCH;
                    off = u == 0 || lg / NG == u ? o : off;
                }
            }
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                const vec xv = *reinterpret_cast<const vec *>(&xs[base[q] + off]);
#pragma unroll
                for (int m = 0; m < NM; ++m) acc[m][q] = OP::mma(wa[m], xv, acc[m][q]);
            }
#pragma unroll
            for (int m = 0; m < NM; ++m) wa[m] = wb[m];
        }
    }
#pragma unroll
    for (int q = 0; q < NP; ++q) {
        const int p = (wave * NP + q) * 16 + li;
        const int x = x0 + p % TX, y = y0 + (p / TX) % TY, z = z0 + p / (TX * TY);
        if (x >= g.W || y >= g.H || z >= g.D) continue;
        float *dst = Y + ((int64_t)z * g.H + y) * g.W + x;
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int c = 16 * (mt0 + m) + 4 * lg + v;
                if (c >= co) continue;
                const float val = acc[m][q][v] + (bias ? bias[c] : 0.0f);
                dst[(int64_t)c * g.P] = accumulate ? dst[(int64_t)c * g.P] + val : val;
            }
    }
}

// Weight gradient: a workgroup adds up, over its range of TX x TY x 4 position
// tiles, the products of 16 NM output channels' dY with 16 input channels at
// every tap (the reduction runs over positions).  Its 4 waves take 7 taps each
// (KS = 1: a quarter of the positions each, partial 4 split + wave).  The
// positions of a vector must be consecutive and 16-byte aligned at every tap:
// in BF16 the X stage holds three copies shifted by one x, in FP32 the elements
// are read one by one (4-byte aligned).  Rows are staged with their halo; the
// pitch of a channel keeps 16 channels on distinct banks.  Positions outside
// the grid are zero in both operands.  The FP32 dY values are summed on the way
// for the bias gradient.
// partial[(split KT + tap) co + m][ci], bpart[split][co].
// Measured (64^3 network, BF16): the 15 weight gradients of a pass with their
// bias gradients and reductions 3.7 ms before, 0.72 ms now.
template <typename OP, int KS, int TX, int NM>
__global__ __launch_bounds__(256) void conv_wgrad_kernel(const float *__restrict__ X, int ci,
                                                         Geo g, const float *__restrict__ dY,
                                                         int co, int ntx, int nty, int ntiles,
                                                         int nsplit, float *__restrict__ partial,
                                                         float *__restrict__ bpart) {
    typedef typename OP::elem elem;
    typedef typename OP::vec vec;
    constexpr int VE = OP::VE, KT = KS * KS * KS, PAD = KS / 2;
    constexpr bool BF = VE == 8;
    constexpr int TY = 64 / TX, TZ = 4;       // 256 positions
    constexpr int HX = TX + KS - 1, HY = TY + KS - 1, HZ = TZ + KS - 1, ROWS = HY * HZ;
    constexpr int RP = BF ? TX : HX;          // row pitch of a stage copy
    constexpr int CP = BF ? ROWS * TX + 8 : ROWS * HX + 1;  // channel pitch
    constexpr int NC = BF ? KS : 1;           // stage copies
    constexpr int DP = 256 + VE;              // dY pitch
    constexpr int NSTEP = 64 / VE;            // steps of 4 VE positions per tile
    constexpr int TW = KS == 3 ? 7 : 1;       // taps per wave
    __shared__ __align__(16) elem xs[NC * 16 * CP];
    __shared__ __align__(16) elem ds[16 * NM * DP];
    __shared__ float red[4][16 * NM];
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int c0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * NM, split = blockIdx.z;
    int toff[TW];
#pragma unroll
    for (int q = 0; q < TW; ++q) {
        const int tap = KS == 3 ? (wave * TW + q < KT ? wave * TW + q : KT - 1) : 0;
        const int dz = tap / 9, dy = (tap / 3) % 3, dx = tap % 3;
        toff[q] = KS == 3 ? (dz * HY + dy) * RP + (BF ? dx * 16 * CP : dx) : 0;
    }
    // this lane's vector of a step: BF16 8 positions (TX = 16: half a row,
    // TX = 8: a row), FP32 4 positions
    const int lrow = BF ? (TX == 16 ? lg >> 1 : lg) : (TX == 16 ? 0 : lg >> 1);
    const int lx = BF ? (TX == 16 ? 8 * (lg & 1) : 0) : (TX == 16 ? 4 * lg : 4 * (lg & 1));
    const elem *xb = xs + li * CP + lrow * RP + lx;
    const elem *db = ds + li * DP + lg * VE;
    f4v acc[TW][NM];
    float bsum[16 * NM];
#pragma unroll
    for (int q = 0; q < TW; ++q)
#pragma unroll
        for (int m = 0; m < NM; ++m) acc[q][m] = f4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < 16 * NM; ++m) bsum[m] = 0.0f;
    const int tb = (int)((int64_t)ntiles * split / nsplit),
              te = (int)((int64_t)ntiles * (split + 1) / nsplit);
    for (int tile = tb; tile < te; ++tile) {
        int b = tile;
        const int x0 = (b % ntx) * TX;
        b /= ntx;
        const int y0 = (b % nty) * TY, z0 = (b / nty) * TZ;
        if (tile > tb) __syncthreads();
        {  // dY: thread t's position, every output channel
            const int x = x0 + t % TX, y = y0 + (t / TX) % TY, z = z0 + t / (TX * TY);
            const bool in = x < g.W && y < g.H && z < g.D;
            const int64_t o = in ? ((int64_t)z * g.H + y) * g.W + x : 0;
            float f[16 * NM];
#pragma unroll
            for (int m = 0; m < 16 * NM; ++m)
                f[m] = dY[m0 + m < co ? (int64_t)(m0 + m) * g.P + o : 0];
#pragma unroll
            for (int m = 0; m < 16 * NM; ++m) {
                const float v = in && m0 + m < co ? f[m] : 0.0f;
                bsum[m] += v;
                ds[m * DP + t] = OP::cvt(v);
            }
        }
        constexpr int NE = 16 * ROWS * HX, UE = 8;
        for (int e0 = t; e0 < NE; e0 += 256 * UE) {  // UE loads in flight per thread
            float f[UE];
#pragma unroll
            for (int i = 0; i < UE; ++i) {
                const int e = e0 + 256 * i;
                const int xx = e % HX, r = (e / HX) % ROWS, c = e / (HX * ROWS);
                const int x = x0 + xx - PAD, y = y0 + r % HY - PAD, z = z0 + r / HY - PAD;
                const bool in = e < NE && c0 + c < ci && x >= 0 && x < g.W && y >= 0 &&
                                y < g.H && z >= 0 && z < g.D;
                f[i] = X[in ? (int64_t)(c0 + c) * g.P + ((int64_t)z * g.H + y) * g.W + x : 0];
                f[i] = in ? f[i] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < UE; ++i) {
                const int e = e0 + 256 * i;
                if (e >= NE) break;
                const int xx = e % HX, r = (e / HX) % ROWS, c = e / (HX * ROWS);
                const elem v = OP::cvt(f[i]);
                if constexpr (BF) {
#pragma unroll
                    for (int d = 0; d < KS; ++d)
                        if (xx >= d && xx - d < TX) xs[d * 16 * CP + c * CP + r * TX + xx - d] = v;
                } else {
                    xs[c * CP + r * HX + xx] = v;
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < NSTEP; ++s) {
            if (KS == 1 && (s & 3) != wave) continue;
            // first row of the step: 4 VE / TX rows per step, TY rows per plane
            constexpr int RS = 4 * VE / TX;
            const int off = ((s * RS / TY) * HY + (s * RS) % TY) * RP;
            vec a[NM];
#pragma unroll
            for (int m = 0; m < NM; ++m)
                a[m] = *reinterpret_cast<const vec *>(db + 16 * m * DP + s * 4 * VE);
#pragma unroll
            for (int q = 0; q < TW; ++q) {
                vec v;
                if constexpr (BF) {
                    v = *reinterpret_cast<const vec *>(xb + off + toff[q]);
                } else {
#pragma unroll
                    for (int u = 0; u < VE; ++u) v[u] = xb[off + toff[q] + u];
                }
#pragma unroll
                for (int m = 0; m < NM; ++m) acc[q][m] = OP::mma(a[m], v, acc[q][m]);
            }
        }
    }
    const int pidx = KS == 3 ? split : 4 * split + wave;
#pragma unroll
    for (int q = 0; q < TW; ++q) {
        const int tap = KS == 3 ? wave * TW + q : 0;
        if (tap >= KT || c0 + li >= ci) continue;
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int mm = m0 + 16 * m + 4 * lg + v;
                if (mm < co)
                    partial[(((int64_t)pidx * KT + tap) * co + mm) * ci + c0 + li] = acc[q][m][v];
            }
    }
    if (blockIdx.x != 0 || !bpart) return;
#pragma unroll
    for (int m = 0; m < 16 * NM; ++m) {
        float v = bsum[m];
#pragma unroll
        for (int h = 32; h > 0; h >>= 1) v += __shfl_xor(v, h);
        if (lane == 0) red[wave][m] = v;
    }
    __syncthreads();
    if (t < 16 * NM && m0 + t < co)
        bpart[(int64_t)split * co + m0 + t] = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
}

// dW[(m ci + c) KT + tap] (=|+=) sum_s partial[s][tap][m][c] and, in the blocks
// after nbw, db[m] (=|+=) sum_s bpart[s][m].  64 entries a block; 4 threads an
// entry add every fourth partial and are summed in order (the loop of one
// thread over all partials took 38 us a layer).
__global__ __launch_bounds__(256) void conv_reduce_kernel(const float *__restrict__ partial,
                                                          int np, int KT, int co, int ci,
                                                          float *__restrict__ dW, int nbw,
                                                          const float *__restrict__ bpart, int nb,
                                                          float *__restrict__ db, int accumulate) {
    __shared__ float red[4][64];
    const bool w = (int)blockIdx.x < nbw;
    const int64_t n = w ? (int64_t)KT * co * ci : co;
    const int cnt = w ? np : nb;
    const float *src = w ? partial : bpart;
    const int64_t e = (int64_t)(w ? blockIdx.x : blockIdx.x - nbw) * 64 + (threadIdx.x & 63);
    const int part = threadIdx.x >> 6;
    float s = 0.0f;
    if (e < n) {
#pragma unroll 8
        for (int k = part; k < cnt; k += 4) s += src[(int64_t)k * n + e];
    }
    red[part][threadIdx.x & 63] = s;
    __syncthreads();
    if (part != 0 || e >= n) return;
    const int i = threadIdx.x & 63;
    s = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
    float *dst = db + e;
    if (w) {
        const int64_t c = e % ci, r = e / ci, m = r % co, tap = r / co;
        dst = dW + (m * ci + c) * KT + tap;
    }
    *dst = accumulate ? *dst + s : s;
}

__global__ __launch_bounds__(256) void leaky_fwd_kernel(float *__restrict__ y, int64_t n,
                                                        float slope) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const float v = y[i];
        y[i] = v > 0.0f ? v : slope * v;
    }
}

// dy *= (y > 0 ? 1 : slope), y the activation's output
__global__ __launch_bounds__(256) void leaky_bwd_kernel(const float *__restrict__ y,
                                                        float *__restrict__ dy, int64_t n,
                                                        float slope) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        dy[i] = y[i] > 0.0f ? dy[i] : slope * dy[i];
}

// coarse[c][z][y][x] = mean of the 2x2x2 fine children (fine dims 2D x 2H x 2W)
__global__ __launch_bounds__(256) void pool_fwd_kernel(const float *__restrict__ fine, int c,
                                                       Geo cg, float *__restrict__ coarse) {
    const int64_t total = (int64_t)c * cg.P;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t ch = i / cg.P, p = i % cg.P;
        const int x = (int)(p % cg.W);
        const int64_t r = p / cg.W;
        const int y = (int)(r % cg.H), z = (int)(r / cg.H);
        const int W2 = 2 * cg.W, H2 = 2 * cg.H;
        const float *f = fine + ch * 8 * cg.P;
        float s = 0.0f;
        for (int q = 0; q < 8; ++q)
            s += f[((int64_t)(2 * z + (q >> 2)) * H2 + 2 * y + ((q >> 1) & 1)) * W2 + 2 * x +
                   (q & 1)];
        coarse[i] = 0.125f * s;
    }
}

// fine (=|+=) coarse / 8 (pool backward) or coarse (upsample forward), by fine index
__global__ __launch_bounds__(256) void spread_kernel(const float *__restrict__ coarse, int c,
                                                     Geo fg, float scale,
                                                     float *__restrict__ fine, int accumulate) {
    const int64_t total = (int64_t)c * fg.P;
    const int Wc = fg.W / 2, Hc = fg.H / 2;
    const int64_t Pc = fg.P / 8;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t ch = i / fg.P, p = i % fg.P;
        const int x = (int)(p % fg.W);
        const int64_t r = p / fg.W;
        const int y = (int)(r % fg.H), z = (int)(r / fg.H);
        const float v =
            scale * coarse[ch * Pc + ((int64_t)(z >> 1) * Hc + (y >> 1)) * Wc + (x >> 1)];
        fine[i] = accumulate ? fine[i] + v : v;
    }
}

// coarse (=|+=) sum of the 8 fine children (upsample backward)
__global__ __launch_bounds__(256) void gather8_kernel(const float *__restrict__ fine, int c,
                                                      Geo cg, float *__restrict__ coarse,
                                                      int accumulate) {
    const int64_t total = (int64_t)c * cg.P;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t ch = i / cg.P, p = i % cg.P;
        const int x = (int)(p % cg.W);
        const int64_t r = p / cg.W;
        const int y = (int)(r % cg.H), z = (int)(r / cg.H);
        const int W2 = 2 * cg.W, H2 = 2 * cg.H;
        const float *f = fine + ch * 8 * cg.P;
        float s = 0.0f;
        for (int q = 0; q < 8; ++q)
            s += f[((int64_t)(2 * z + (q >> 2)) * H2 + 2 * y + ((q >> 1) & 1)) * W2 + 2 * x +
                   (q & 1)];
        coarse[i] = accumulate ? coarse[i] + s : s;
    }
}

// per-block sums of (y - t)^2; dy = 2 (y - t) / n
__global__ __launch_bounds__(256) void mse_kernel(const float *__restrict__ y,
                                                  const float *__restrict__ tg, int64_t n,
                                                  float *__restrict__ dy,
                                                  double *__restrict__ partial) {
    __shared__ double red[256];
    double s = 0.0;
    const float sc = 2.0f / (float)n;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const float d = y[i] - tg[i];
        s += (double)d * d;
        if (dy) dy[i] = sc * d;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void adam_kernel(float *__restrict__ p,
                                                   const float *__restrict__ g,
                                                   float *__restrict__ m, float *__restrict__ v,
                                                   int64_t n, float lr, float b1, float b2,
                                                   float eps, float c1, float c2) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi * c1) / (sqrtf(vi * c2) + eps);
    }
}

__global__ __launch_bounds__(256) void f64_to_f32_scaled(const double *__restrict__ s,
                                                         float *__restrict__ d, int64_t n,
                                                         double scale) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        d[i] = (float)(s[i] * scale);
}

__global__ __launch_bounds__(256) void f32_to_f64_scaled(const float *__restrict__ s,
                                                         double *__restrict__ d, int64_t n,
                                                         double scale) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x)
        d[i] = (double)s[i] * scale;
}

unsigned nblk(int64_t n) {
    return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 65536));
}

int make_geo(const int32_t dims[3], Geo &g) {
    TT_CHECK(dims && dims[0] > 0 && dims[1] > 0 && dims[2] > 0, TTDFT_EBADARG,
             "nn: bad spatial dims");
    g.D = dims[0];
    g.H = dims[1];
    g.W = dims[2];
    g.P = (int64_t)g.D * g.H * g.W;
    return TTDFT_OK;
}

int tiles_of(int n, int t) { return (n + t - 1) / t; }

template <typename OP, int KS, int NG, int TX, int TY, int TZ, int NM>
void conv_launch(ttdft_ctx ctx, const float *x, int ci, const Geo &g,
                 const typename OP::elem *wf, const float *b, int co, float *y, int accumulate,
                 int nchunk) {
    const int ntx = tiles_of(g.W, TX), nty = tiles_of(g.H, TY), ntz = tiles_of(g.D, TZ);
    hipLaunchKernelGGL((conv_kernel<OP, KS, NG, TX, TY, TZ, NM>),
                       dim3((unsigned)(ntx * nty * ntz), (unsigned)tiles_of(co, 16 * NM)),
                       dim3(256), 0, ctx->stream, x, ci, g, wf, b, co, y, accumulate, nchunk, ntx,
                       nty);
}

// Position tile and row tiles per workgroup.  Large grids take 256 positions
// (a 16 x 4 x 4 tile, or 8 x 8 x 4 where x pads less) and up to 64 output
// channels, so that a staged halo serves the most products; where that leaves
// fewer than 256 workgroups (one per CU) tiles of 64 positions (8 x 4 x 2) and
// 32 or 16 channels spread the work.
template <typename OP, int KS, int NG>
void conv_shape(ttdft_ctx ctx, const float *x, int ci, const Geo &g,
                const typename OP::elem *wf, const float *b, int co, float *y, int accumulate,
                int nchunk) {
    const int mt = tiles_of(co, 16);
    const bool wide = tiles_of(g.W, 16) * 16 <= tiles_of(g.W, 8) * 8;
    const int64_t big = wide ? (int64_t)tiles_of(g.W, 16) * tiles_of(g.H, 4) * tiles_of(g.D, 4)
                             : (int64_t)tiles_of(g.W, 8) * tiles_of(g.H, 8) * tiles_of(g.D, 4);
    const int64_t small = (int64_t)tiles_of(g.W, 8) * tiles_of(g.H, 4) * tiles_of(g.D, 2);
#define CONV(TX, TY, TZ, NM) \
    conv_launch<OP, KS, NG, TX, TY, TZ, NM>(ctx, x, ci, g, wf, b, co, y, accumulate, nchunk)
    const int nm = mt >= 3 ? 4 : mt;
    if (big * tiles_of(mt, nm) >= 256) {
        if (wide && nm == 4) CONV(16, 4, 4, 4);
        else if (wide && nm == 2) CONV(16, 4, 4, 2);
        else if (wide) CONV(16, 4, 4, 1);
        else if (nm == 4) CONV(8, 8, 4, 4);
        else if (nm == 2) CONV(8, 8, 4, 2);
        else CONV(8, 8, 4, 1);
    } else if (mt >= 2 && small * tiles_of(mt, 2) >= 256) {
        CONV(8, 4, 2, 2);
    } else {
        CONV(8, 4, 2, 1);
    }
#undef CONV
}

// flip: the data gradient (x = dY, its ci outputs are the layer's inputs)
template <typename OP>
int conv_run(ttdft_ctx ctx, const float *x, int ci, const Geo &g, const float *w, int flip,
             const float *b, int co, int ks, float *y, int accumulate) {
    const int KT = ks * ks * ks;
    // channel vectors per position and chunk: four, or two where that pads fewer
    // channels (16 or 48 channels in BF16)
    const int c4 = tiles_of(ci, 4 * OP::VE) * 4, c2 = tiles_of(ci, 2 * OP::VE) * 2;
    const int NG = ks == 3 && c2 < c4 ? 2 : 4;
    const int nchunk = tiles_of(ci, NG * OP::VE), nsteps = (KT * NG + 3) / 4;
    // row tiles up to a workgroup's full group of four: the last group reads
    // whole tiles
    const int mt = tiles_of(co, 64) * 4;
    const int64_t total = (int64_t)mt * nchunk * nsteps * 64;
    TT_CHECK((total + 255) / 256 < (1LL << 31) && tiles_of(co, 32) <= 65535, TTDFT_EBADARG,
             "conv3d: layer too large (%d -> %d channels)", ci, co);
    TT_TRY(ctx->nn_scratch[0].ensure((size_t)total * 16));
    typename OP::elem *wf = (typename OP::elem *)ctx->nn_scratch[0].ptr;
    hipLaunchKernelGGL((conv_weights_kernel<OP>), dim3((unsigned)((total + 255) / 256)),
                       dim3(256), 0, ctx->stream, w, co, ci, KT, flip, NG, nchunk, nsteps,
                       total, wf);
    TT_LAUNCH_CHECK();
    if (ks == 1)
        conv_shape<OP, 1, 4>(ctx, x, ci, g, wf, b, co, y, accumulate, nchunk);
    else if (NG == 2)
        conv_shape<OP, 3, 2>(ctx, x, ci, g, wf, b, co, y, accumulate, nchunk);
    else
        conv_shape<OP, 3, 4>(ctx, x, ci, g, wf, b, co, y, accumulate, nchunk);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int conv_forward(ttdft_ctx ctx, const float *x, int ci, const Geo &g, const float *w, int flip,
                 const float *b, int co, int ks, float *y, int accumulate) {
    return ctx->nn_math == TTDFT_NN_BF16
               ? conv_run<Bf16Op>(ctx, x, ci, g, w, flip, b, co, ks, y, accumulate)
               : conv_run<F32Op>(ctx, x, ci, g, w, flip, b, co, ks, y, accumulate);
}

template <typename OP, int KS, int TX, int NM>
void wgrad_launch(ttdft_ctx ctx, const float *x, int ci, const Geo &g, const float *dy, int co,
                  int nsplit, float *partial, float *bpart) {
    constexpr int TY = 64 / TX;
    const int ntx = tiles_of(g.W, TX), nty = tiles_of(g.H, TY), ntz = tiles_of(g.D, 4);
    hipLaunchKernelGGL((conv_wgrad_kernel<OP, KS, TX, NM>),
                       dim3((unsigned)tiles_of(ci, 16), (unsigned)tiles_of(co, 16 * NM),
                            (unsigned)nsplit),
                       dim3(256), 0, ctx->stream, x, ci, g, dy, co, ntx, nty, ntx * nty * ntz,
                       nsplit, partial, bpart);
}

template <typename OP>
int wgrad_run(ttdft_ctx ctx, const float *x, int ci, const Geo &g, const float *dy, int co, int ks,
              float *dw, float *db, int accumulate) {
    const int KT = ks * ks * ks;
    // x extent of a position tile: 16, or 8 where that pads less; 32 output
    // channels per workgroup when the layer has them; position ranges for about
    // two workgroups per CU
    const bool wide = tiles_of(g.W, 16) * 16 <= tiles_of(g.W, 8) * 8;
    const int nm = co > 16 ? 2 : 1;
    const int64_t ntiles = wide
                               ? (int64_t)tiles_of(g.W, 16) * tiles_of(g.H, 4) * tiles_of(g.D, 4)
                               : (int64_t)tiles_of(g.W, 8) * tiles_of(g.H, 8) * tiles_of(g.D, 4);
    const int64_t wgs = (int64_t)tiles_of(ci, 16) * tiles_of(co, 16 * nm);
    const int nsplit = (int)std::max<int64_t>(1, std::min<int64_t>((512 + wgs - 1) / wgs, ntiles));
    const int np = ks == 3 ? nsplit : 4 * nsplit;
    const int64_t nw = (int64_t)co * ci * KT;
    TT_TRY(ctx->nn_scratch[1].ensure(sizeof(float) * ((size_t)nw * np + (size_t)co * nsplit)));
    float *partial = (float *)ctx->nn_scratch[1].ptr, *bpart = partial + nw * np;
    float *bp = db ? bpart : nullptr;
#define WGRAD(KS, TX, NM) wgrad_launch<OP, KS, TX, NM>(ctx, x, ci, g, dy, co, nsplit, partial, bp)
    if (ks == 3) {
        if (wide && nm == 2) WGRAD(3, 16, 2);
        else if (wide) WGRAD(3, 16, 1);
        else if (nm == 2) WGRAD(3, 8, 2);
        else WGRAD(3, 8, 1);
    } else {
        if (wide && nm == 2) WGRAD(1, 16, 2);
        else if (wide) WGRAD(1, 16, 1);
        else if (nm == 2) WGRAD(1, 8, 2);
        else WGRAD(1, 8, 1);
    }
#undef WGRAD
    TT_LAUNCH_CHECK();
    const int nbw = (int)((nw + 63) / 64), nbb = db ? tiles_of(co, 64) : 0;
    hipLaunchKernelGGL(conv_reduce_kernel, dim3((unsigned)(nbw + nbb)), dim3(256), 0, ctx->stream,
                       partial, np, KT, co, ci, dw, nbw, bpart, nsplit, db, accumulate);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int check_conv(ttdft_ctx ctx, int ci, int co, int ks) {
    TT_CHECK(ctx, TTDFT_EBADARG, "nn: NULL context");
    TT_CHECK(ci >= 1 && co >= 1 && (ks == 1 || ks == 3), TTDFT_EBADARG,
             "conv3d: channels %d -> %d, kernel %d (1 or 3)", ci, co, ks);
    TT_CHECK((int64_t)ci * ks * ks * ks < (1 << 30), TTDFT_EBADARG, "conv3d: too many inputs");
    return TTDFT_OK;
}

}  // namespace
}  // namespace ttdft

using namespace ttdft;

extern "C" {

int ttdft_nn_set_math(ttdft_ctx ctx, int math) {
    clear_error();
    TT_CHECK(ctx && (math == TTDFT_NN_FP32 || math == TTDFT_NN_BF16), TTDFT_EBADARG,
             "nn_set_math: unknown mode %d", math);
    ctx->nn_math = math;
    return TTDFT_OK;
}

int ttdft_nn_conv3d_forward(ttdft_ctx ctx, const float *d_x, int32_t ci, const int32_t dims[3],
                            const float *d_w, const float *d_b, int32_t co, int32_t ks,
                            float *d_y, int accumulate) {
    clear_error();
    TT_TRY(check_conv(ctx, ci, co, ks));
    Geo g;
    TT_TRY(make_geo(dims, g));
    TT_CHECK(d_x && d_w && d_y, TTDFT_EBADARG, "conv3d_forward: NULL tensor");
    TT_HIP(hipSetDevice(ctx->device));
    return conv_forward(ctx, d_x, ci, g, d_w, 0, d_b, co, ks, d_y, accumulate);
}

int ttdft_nn_conv3d_backward_data(ttdft_ctx ctx, const float *d_dy, int32_t co,
                                  const int32_t dims[3], const float *d_w, int32_t ci,
                                  int32_t ks, float *d_dx, int accumulate) {
    clear_error();
    TT_TRY(check_conv(ctx, ci, co, ks));
    Geo g;
    TT_TRY(make_geo(dims, g));
    TT_CHECK(d_dy && d_w && d_dx, TTDFT_EBADARG, "conv3d_backward_data: NULL tensor");
    TT_HIP(hipSetDevice(ctx->device));
    return conv_forward(ctx, d_dy, co, g, d_w, 1, nullptr, ci, ks, d_dx, accumulate);
}

int ttdft_nn_conv3d_backward_weight(ttdft_ctx ctx, const float *d_x, int32_t ci,
                                    const int32_t dims[3], const float *d_dy, int32_t co,
                                    int32_t ks, float *d_dw, float *d_db, int accumulate) {
    clear_error();
    TT_TRY(check_conv(ctx, ci, co, ks));
    Geo g;
    TT_TRY(make_geo(dims, g));
    TT_CHECK(d_x && d_dy && d_dw, TTDFT_EBADARG, "conv3d_backward_weight: NULL tensor");
    TT_HIP(hipSetDevice(ctx->device));
    return ctx->nn_math == TTDFT_NN_BF16
               ? wgrad_run<Bf16Op>(ctx, d_x, ci, g, d_dy, co, ks, d_dw, d_db, accumulate)
               : wgrad_run<F32Op>(ctx, d_x, ci, g, d_dy, co, ks, d_dw, d_db, accumulate);
}

int ttdft_nn_leaky_relu(ttdft_ctx ctx, float *d_y, int64_t n, float slope) {
    clear_error();
    TT_CHECK(ctx && d_y && n >= 0, TTDFT_EBADARG, "leaky_relu: bad arguments");
    if (n == 0) return TTDFT_OK;
    TT_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(leaky_fwd_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream, d_y, n, slope);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int ttdft_nn_leaky_relu_backward(ttdft_ctx ctx, const float *d_y, float *d_dy, int64_t n,
                                 float slope) {
    clear_error();
    TT_CHECK(ctx && d_y && d_dy && n >= 0, TTDFT_EBADARG, "leaky_relu_backward: bad arguments");
    if (n == 0) return TTDFT_OK;
    TT_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(leaky_bwd_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream, d_y, d_dy, n,
                       slope);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int ttdft_nn_avgpool2(ttdft_ctx ctx, const float *d_fine, int32_t c, const int32_t fine_dims[3],
                      float *d_coarse) {
    clear_error();
    Geo f;
    TT_TRY(make_geo(fine_dims, f));
    TT_CHECK(ctx && d_fine && d_coarse && c >= 1 && f.D % 2 == 0 && f.H % 2 == 0 && f.W % 2 == 0,
             TTDFT_EBADARG, "avgpool2: bad arguments (even dims needed)");
    TT_HIP(hipSetDevice(ctx->device));
    const int32_t cd[3] = {f.D / 2, f.H / 2, f.W / 2};
    Geo cg;
    TT_TRY(make_geo(cd, cg));
    hipLaunchKernelGGL(pool_fwd_kernel, dim3(nblk(c * cg.P)), dim3(256), 0, ctx->stream, d_fine,
                       c, cg, d_coarse);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int ttdft_nn_avgpool2_backward(ttdft_ctx ctx, const float *d_dcoarse, int32_t c,
                               const int32_t fine_dims[3], float *d_dfine, int accumulate) {
    clear_error();
    Geo f;
    TT_TRY(make_geo(fine_dims, f));
    TT_CHECK(ctx && d_dcoarse && d_dfine && c >= 1 && f.D % 2 == 0 && f.H % 2 == 0 &&
                 f.W % 2 == 0,
             TTDFT_EBADARG, "avgpool2_backward: bad arguments (even dims needed)");
    TT_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(spread_kernel, dim3(nblk(c * f.P)), dim3(256), 0, ctx->stream, d_dcoarse,
                       c, f, 0.125f, d_dfine, accumulate);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int ttdft_nn_upsample2(ttdft_ctx ctx, const float *d_coarse, int32_t c,
                       const int32_t fine_dims[3], float *d_fine) {
    clear_error();
    Geo f;
    TT_TRY(make_geo(fine_dims, f));
    TT_CHECK(ctx && d_coarse && d_fine && c >= 1 && f.D % 2 == 0 && f.H % 2 == 0 && f.W % 2 == 0,
             TTDFT_EBADARG, "upsample2: bad arguments (even dims needed)");
    TT_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(spread_kernel, dim3(nblk(c * f.P)), dim3(256), 0, ctx->stream, d_coarse, c,
                       f, 1.0f, d_fine, 0);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int ttdft_nn_upsample2_backward(ttdft_ctx ctx, const float *d_dfine, int32_t c,
                                const int32_t fine_dims[3], float *d_dcoarse, int accumulate) {
    clear_error();
    Geo f;
    TT_TRY(make_geo(fine_dims, f));
    TT_CHECK(ctx && d_dfine && d_dcoarse && c >= 1 && f.D % 2 == 0 && f.H % 2 == 0 &&
                 f.W % 2 == 0,
             TTDFT_EBADARG, "upsample2_backward: bad arguments (even dims needed)");
    TT_HIP(hipSetDevice(ctx->device));
    const int32_t cd[3] = {f.D / 2, f.H / 2, f.W / 2};
    Geo cg;
    TT_TRY(make_geo(cd, cg));
    hipLaunchKernelGGL(gather8_kernel, dim3(nblk(c * cg.P)), dim3(256), 0, ctx->stream, d_dfine,
                       c, cg, d_dcoarse, accumulate);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int ttdft_nn_mse(ttdft_ctx ctx, const float *d_y, const float *d_t, int64_t n, float *d_dy,
                 double *loss) {
    clear_error();
    TT_CHECK(ctx && d_y && d_t && n > 0 && loss, TTDFT_EBADARG, "mse: bad arguments");
    TT_HIP(hipSetDevice(ctx->device));
    constexpr int kBlocks = 512;
    TT_TRY(ctx->scratch[6].ensure(sizeof(double) * kBlocks));
    double *partial = (double *)ctx->scratch[6].ptr;
    hipLaunchKernelGGL(mse_kernel, dim3(kBlocks), dim3(256), 0, ctx->stream, d_y, d_t, n, d_dy,
                       partial);
    TT_LAUNCH_CHECK();
    std::vector<double> h(kBlocks);
    TT_HIP(hipMemcpyAsync(h.data(), partial, sizeof(double) * kBlocks, hipMemcpyDeviceToHost,
                          ctx->stream));
    TT_HIP(hipStreamSynchronize(ctx->stream));
    double s = 0.0;
    for (double v : h) s += v;
    *loss = s / (double)n;
    return TTDFT_OK;
}

int ttdft_nn_adam(ttdft_ctx ctx, float *d_p, const float *d_g, float *d_m, float *d_v, int64_t n,
                  float lr, float beta1, float beta2, float eps, int32_t step) {
    clear_error();
    TT_CHECK(ctx && d_p && d_g && d_m && d_v && n >= 0 && step >= 1, TTDFT_EBADARG,
             "adam: bad arguments");
    if (n == 0) return TTDFT_OK;
    TT_HIP(hipSetDevice(ctx->device));
    const float c1 = (float)(1.0 / (1.0 - std::pow((double)beta1, step)));
    const float c2 = (float)(1.0 / (1.0 - std::pow((double)beta2, step)));
    hipLaunchKernelGGL(adam_kernel, dim3(nblk(n)), dim3(256), 0, ctx->stream, d_p, d_g, d_m, d_v,
                       n, lr, beta1, beta2, eps, c1, c2);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int ttdft_nn_to_f32(ttdft_ctx ctx, const double *d_src, float *d_dst, int64_t n, double scale) {
    clear_error();
    TT_CHECK(ctx && d_src && d_dst && n >= 0, TTDFT_EBADARG, "to_f32: bad arguments");
    if (n == 0) return TTDFT_OK;
    TT_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(f64_to_f32_scaled, dim3(nblk(n)), dim3(256), 0, ctx->stream, d_src, d_dst,
                       n, scale);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

int ttdft_nn_to_f64(ttdft_ctx ctx, const float *d_src, double *d_dst, int64_t n, double scale) {
    clear_error();
    TT_CHECK(ctx && d_src && d_dst && n >= 0, TTDFT_EBADARG, "to_f64: bad arguments");
    if (n == 0) return TTDFT_OK;
    TT_HIP(hipSetDevice(ctx->device));
    hipLaunchKernelGGL(f32_to_f64_scaled, dim3(nblk(n)), dim3(256), 0, ctx->stream, d_src, d_dst,
                       n, scale);
    TT_LAUNCH_CHECK();
    return TTDFT_OK;
}

}  // extern "C"
