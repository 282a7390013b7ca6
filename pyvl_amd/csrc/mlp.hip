// Small MLP (BF16 operands, FP32 accumulation) trained and evaluated on the GPU with
// hand-written kernels: it predicts each panel's circulation to warm-start the iterative
// solve.  No reference counterpart (the reference solves every step with LAPACK).
//
// Network: in -> W1 -> SiLU -> W2 -> SiLU -> ... -> W_L -> out (scalar), width 256.
// Parameters are kept in FP32 (master copy, Adam moments) and mirrored in BF16 for the
// products.  Activations and back-propagated errors are stored in BF16; every product
// accumulates in FP32 on v_mfma_f32_16x16x32_bf16.
#include "pvl_internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

using namespace pvl;

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct pvl_mlp
{
    int d_in = 0, width = 0, n_layers = 0;
    std::vector<int> dims;          // n_layers + 1 entries
    std::vector<size_t> w_off, b_off; // offsets into the flat parameter vector
    size_t n_params = 0;
    float *d_p = nullptr, *d_g = nullptr, *d_m = nullptr, *d_v = nullptr; // FP32 master, grad, Adam
    bf16 *d_pb = nullptr;           // BF16 mirror
    int cap_batch = 0, cap_general = 0; // samples that the batch buffers hold (ensure_batch, ensure_general)
    std::vector<bf16 *> d_act;      // [n_layers] layer inputs A_l (batch x dims[l]) in BF16
    std::vector<float *> d_z;       // [n_layers] pre-activations Z_l (batch x dims[l+1]) FP32
    std::vector<bf16 *> d_delta;    // [n_layers] error of each layer's output (batch x dims[l+1])
    float *d_part = nullptr;        // [kMaxSplits][n_params] gradient sums per slice of the batch
    float *d_loss_part = nullptr;   // per workgroup of the fused pass
    float *d_loss = nullptr;        // 1
    bf16 *d_pt = nullptr;           // transposed BF16 mirror of the hidden layers' weights
    bool pt_valid = false;          // refreshed at the first backward pass after a change
    long step = 0;
};

namespace
{

__device__ __forceinline__ float silu(float z) { return z / (1.0f + __expf(-z)); }
__device__ __forceinline__ float silu_grad(float z)
{
    const float s = 1.0f / (1.0f + __expf(-z));
    return s * (1.0f + z * (1.0f - s));
}

// C[m][j] = sum_r A(m, r) * B(j, r) with A(m, r) = A[m*am + r*ar], B(j, r) = B[j*bj + r*br]
// (BF16 operands, FP32 accumulation on MFMA 16x16x32).  64x64 tile per workgroup, 32x32
// per wave; K staged through LDS in steps of 32.  Epilogues:
//   EPI_FWD:  Z = C + bias[j] (FP32 out), Anext = SiLU(Z) in BF16 (if act) or Z
//   EPI_BWD:  D = C * SiLU'(Zprev[m][j])  -> BF16
//   EPI_WGRAD: G[m][j] = C (FP32)
enum
{
    EPI_FWD = 0,
    EPI_BWD = 1,
    EPI_WGRAD = 2
};

template <int EPI>
__global__ void __launch_bounds__(256) gemm_bf16_kernel(int M, int N, int R, const bf16 *__restrict__ A, long am,
                                                        long ar, const bf16 *__restrict__ B, long bj, long br,
                                                        const float *__restrict__ bias, float *__restrict__ outf,
                                                        bf16 *__restrict__ outb, const float *__restrict__ zprev,
                                                        int act)
{
    constexpr int KS = 32, LD = KS + 8;
    __shared__ bf16 As[64][LD];
    __shared__ bf16 Bs[64][LD];
    const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    const int wm = w >> 1, wn = w & 1, lr = lane & 15, lk = lane >> 4;
    const int m0 = blockIdx.y * 64, j0 = blockIdx.x * 64;
    f32x4 acc[2][2];
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b)
            acc[a][b] = f32x4{0, 0, 0, 0};
    for (int r0 = 0; r0 < R; r0 += KS)
    {
        for (int idx = tid; idx < 64 * KS; idx += 256)
        {
            const int i = idx / KS, k = idx % KS;
            const int m = m0 + i, j = j0 + i, r = r0 + k;
            As[i][k] = (m < M && r < R) ? A[m * am + r * ar] : (bf16)0.0f;
            Bs[i][k] = (j < N && r < R) ? B[j * bj + r * br] : (bf16)0.0f;
        }
        __syncthreads();
        bf16x8 af[2], bfr[2];
        for (int a = 0; a < 2; ++a)
            for (int e = 0; e < 8; ++e)
                af[a][e] = As[32 * wm + 16 * a + lr][8 * lk + e];
        for (int b = 0; b < 2; ++b)
            for (int e = 0; e < 8; ++e)
                bfr[b][e] = Bs[32 * wn + 16 * b + lr][8 * lk + e];
        for (int a = 0; a < 2; ++a)
            for (int b = 0; b < 2; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], bfr[b], acc[a][b], 0, 0, 0);
        __syncthreads();
    }
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b)
            for (int v = 0; v < 4; ++v)
            {
                const int m = m0 + 32 * wm + 16 * a + 4 * lk + v;
                const int j = j0 + 32 * wn + 16 * b + lr;
                if (m >= M || j >= N)
                    continue;
                const float c = acc[a][b][v];
                const long o = (long)m * N + j;
                if constexpr (EPI == EPI_FWD)
                {
                    const float z = c + bias[j];
                    if (outf)
                        outf[o] = z;
                    if (outb)
                        outb[o] = (bf16)(act ? silu(z) : z);
                }
                else if constexpr (EPI == EPI_BWD)
                {
                    outb[o] = (bf16)(c * silu_grad(zprev[o]));
                }
                else
                {
                    outf[o] = c;
                }
            }
}

// ---------------------------------------------------------------------------------------
// Fused pass for networks whose activations fit the LDS (fused_lds_bytes): a workgroup takes
// kRows samples through all layers and, when training, back: inputs, pre-activations and errors
// stay in LDS, weights are read as MFMA operands from L2 (BF16, 16 bytes per lane: row j of W for
// the forward products, row k of W^T, the mirror d_pt, for the backward ones).  What the weight
// gradients need (each layer's input and output error, BF16) is written once.  Products accumulate
// in the same order as in gemm_bf16_kernel, so outputs and errors are the same bit for bit.
// Bound by the chain of layers (weights from L2, products, SiLU, a barrier: ~8 us each) with one
// workgroup per CU; one launch instead of nine (8,192 samples, width 256, four layers, forward and
// backward without the weight gradients: 205 us of kernels -> 45 us).
constexpr int kRows = 32;
constexpr int kFusedWaves = 8, kCt = 2; // column tiles of 16 per wave: 256 columns at once
constexpr int kMaxFusedLayers = 8;
constexpr int kMaxSplits = 16;
struct FusedNet
{
    int n_layers, dims[kMaxFusedLayers + 1];
    const bf16 *w[kMaxFusedLayers], *wt[kMaxFusedLayers]; // W (out x in) and, hidden layers, W^T (in x out)
    const float *bias[kMaxFusedLayers];
    bf16 *act[kMaxFusedLayers];   // act[l]: input of layer l (l >= 1), batch x dims[l]
    bf16 *delta[kMaxFusedLayers]; // batch x dims[l + 1]
};
// row stride of the activations in LDS: the widest input rounded up to an MFMA step, and 16 bytes
// that spread the rows over the banks
constexpr int lds_stride(int width) { return (width + 31) / 32 * 32 + 8; }
size_t fused_lds_bytes(const pvl_mlp *h, bool train)
{
    const size_t ld = lds_stride(std::max(h->width, h->d_in));
    return sizeof(bf16) * 2 * kRows * ld + (train ? sizeof(float) * (size_t)(h->n_layers - 1) * kRows * h->width : 0) +
           sizeof(float) * kRows;
}

// acc[rt][ct] += A B^T over K for the wave's column tiles j0 + 16 ct: A (kRows x K) in LDS, row j
// of B at b + j * K in global memory (K a multiple of 8 and 16-byte rows when VEC).  The operands
// of eight K steps are loaded before the first product: one trip to L2 for 256 inputs.
template <bool VEC>
__device__ __forceinline__ void fused_product(const bf16 *A, int lda, const bf16 *__restrict__ b, int K, int n_cols,
                                              int j0, int lane, f32x4 (&acc)[2][kCt])
{
    constexpr int S = VEC ? 8 : 1;
    const int lr = lane & 15, lk = lane >> 4;
#pragma unroll 1
    for (int r0 = 0; r0 < K; r0 += 32 * S)
    {
        bf16x8 bf[S][kCt];
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int ct = 0; ct < kCt; ++ct)
            {
                const int j = j0 + 16 * ct + lr, k = r0 + 32 * s + 8 * lk;
                if constexpr (VEC)
                {
                    // clamped address, zeroed operand: no branch around the load
                    const bool in = j < n_cols && k < K;
                    const bf16x8 v = *reinterpret_cast<const bf16x8 *>(b + (size_t)min(j, n_cols - 1) * K + min(k, K - 8));
                    bf[s][ct] = in ? v : bf16x8{};
                }
                else
                {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        bf[s][ct][e] = (j < n_cols && k + e < K) ? b[(size_t)j * K + k + e] : (bf16)0.0f;
                }
            }
#pragma unroll
        for (int s = 0; s < S; ++s)
        {
            if (r0 + 32 * s >= K)
                break;
            bf16x8 af[2];
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
                af[rt] = *reinterpret_cast<const bf16x8 *>(A + (16 * rt + lr) * lda + r0 + 32 * s + 8 * lk);
#pragma unroll
            for (int ct = 0; ct < kCt; ++ct)
#pragma unroll
                for (int rt = 0; rt < 2; ++rt)
                    acc[rt][ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[rt], bf[s][ct], acc[rt][ct], 0, 0, 0);
        }
    }
}

// The first `rows` of the workgroup's kRows x W values in LDS to global memory (row-major), 16
// bytes per lane where W allows.
__device__ __forceinline__ void store_rows(bf16 *__restrict__ dst, const bf16 *src, int lds_ld, int W, int rows, int w,
                                           int lane)
{
    if (W % 8 == 0)
    {
        const int per = W / 8, n = min(rows, kRows) * per;
        for (int i = 64 * w + lane; i < n; i += 64 * kFusedWaves)
        {
            const int r = i / per, c = 8 * (i - r * per);
            *reinterpret_cast<bf16x8 *>(dst + (size_t)r * W + c) = *reinterpret_cast<const bf16x8 *>(src + r * lds_ld + c);
        }
    }
    else
        for (int r = w; r < min(rows, kRows); r += kFusedWaves)
            for (int c = lane; c < W; c += 64)
                dst[(size_t)r * W + c] = src[r * lds_ld + c];
}

template <bool TRAIN>
__global__ void __launch_bounds__(64 * kFusedWaves)
    fused_kernel(FusedNet net, const float *__restrict__ X, const float *__restrict__ T, int batch,
                 float *__restrict__ Y, float *__restrict__ loss_part)
{
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int L = net.n_layers, W = net.dims[1], d_in = net.dims[0];
    const int LD = (max(W, d_in) + 31) / 32 * 32 + 8;
    bf16 *a0 = (bf16 *)smem_raw, *a1 = a0 + kRows * LD;
    float *z = (float *)(a1 + kRows * LD); // [L - 1][kRows][W], training
    float *red = z + (TRAIN ? (size_t)(L - 1) * kRows * W : 0);
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m0 = blockIdx.x * kRows;
    // inputs in BF16, zero past the batch and past d_in (and in the padding of every later layer)
    for (int r = w; r < kRows; r += kFusedWaves)
        for (int c = lane; c < LD; c += 64)
        {
            a0[r * LD + c] = (m0 + r < batch && c < d_in) ? (bf16)X[(size_t)(m0 + r) * d_in + c] : (bf16)0.0f;
            a1[r * LD + c] = (bf16)0.0f;
        }
    __syncthreads();
    for (int l = 0; l + 1 < L; ++l)
    {
        const int K = net.dims[l];
        for (int j0 = 16 * kCt * w; j0 < W; j0 += 16 * kCt * kFusedWaves)
        {
            f32x4 acc[2][kCt] = {};
            if (K % 8 == 0)
                fused_product<true>(a0, LD, net.w[l], K, W, j0, lane, acc);
            else
                fused_product<false>(a0, LD, net.w[l], K, W, j0, lane, acc);
#pragma unroll
            for (int ct = 0; ct < kCt; ++ct)
            {
                const int j = j0 + 16 * ct + lr;
                if (j >= W)
                    continue;
                const float bj = net.bias[l][j];
#pragma unroll
                for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                    {
                        const int r = 16 * rt + 4 * lk + v;
                        const float zz = acc[rt][ct][v] + bj;
                        a1[r * LD + j] = (bf16)silu(zz);
                        if constexpr (TRAIN)
                            z[((size_t)l * kRows + r) * W + j] = zz;
                    }
            }
        }
        __syncthreads();
        if constexpr (TRAIN)
            store_rows(net.act[l + 1] + (size_t)m0 * W, a1, LD, W, batch - m0, w, lane);
        // the next layer reads a1; its padding columns are zero, a0's (d_in wider than W) are cleared
        bf16 *t = a0;
        a0 = a1, a1 = t;
        if (l == 0 && d_in > W)
        {
            for (int i = tid; i < kRows * LD; i += 64 * kFusedWaves)
                a1[i] = (bf16)0.0f;
            __syncthreads();
        }
    }
    // output layer (one column): a row tile per wave, the product's other columns zero
    if (w < 2)
    {
        const int K = net.dims[L - 1];
        f32x4 c = {};
        for (int r0 = 0; r0 < K; r0 += 32)
        {
            bf16x8 bf;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                bf[e] = (lr == 0 && r0 + 8 * lk + e < K) ? net.w[L - 1][r0 + 8 * lk + e] : (bf16)0.0f;
            const bf16x8 af = *reinterpret_cast<const bf16x8 *>(a0 + (16 * w + lr) * LD + r0 + 8 * lk);
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf, c, 0, 0, 0);
        }
        if (lr == 0)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int r = 16 * w + 4 * lk + v;
                red[r] = c[v] + net.bias[L - 1][0];
            }
    }
    __syncthreads();
    if constexpr (!TRAIN)
    {
        if (tid < kRows && m0 + tid < batch)
            Y[m0 + tid] = red[tid];
    }
    else
    {
        // loss and the output's error 2 (y - t) / batch
        if (tid < 64)
        {
            const bool live = tid < kRows && m0 + tid < batch;
            const float e = live ? red[tid] - T[m0 + tid] : 0.0f;
            const bf16 d = (bf16)(2.0f * e / (float)batch);
            float s = e * e;
            for (int off = 32; off > 0; off >>= 1)
                s += __shfl_xor(s, off);
            if (tid == 0)
                loss_part[blockIdx.x] = s;
            if (tid < kRows)
                red[tid] = (float)d;
            if (live)
                net.delta[L - 1][m0 + tid] = d;
        }
        __syncthreads();
        // error of the last hidden layer's output: one product per entry
        {
            const float *zl = z + (size_t)(L - 2) * kRows * W;
            for (int c = lane; c < W; c += 64)
            {
                const float wc = (float)net.w[L - 1][c];
                for (int r = w; r < kRows; r += kFusedWaves)
                    a1[r * LD + c] = (bf16)(red[r] * wc * silu_grad(zl[r * W + c]));
            }
        }
        __syncthreads();
        store_rows(net.delta[L - 2] + (size_t)m0 * W, a1, LD, W, batch - m0, w, lane);
        for (int l = L - 2; l > 0; --l)
        {
            // error of layer l - 1's output from that of layer l's (in a1), through W_l
            const float *zl = z + (size_t)(l - 1) * kRows * W;
            for (int j0 = 16 * kCt * w; j0 < W; j0 += 16 * kCt * kFusedWaves)
            {
                f32x4 acc[2][kCt] = {};
                if (W % 8 == 0)
                    fused_product<true>(a1, LD, net.wt[l], W, W, j0, lane, acc);
                else
                    fused_product<false>(a1, LD, net.wt[l], W, W, j0, lane, acc);
#pragma unroll
                for (int ct = 0; ct < kCt; ++ct)
                {
                    const int j = j0 + 16 * ct + lr;
                    if (j >= W)
                        continue;
#pragma unroll
                    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                        for (int v = 0; v < 4; ++v)
                        {
                            const int r = 16 * rt + 4 * lk + v;
                            a0[r * LD + j] = (bf16)(acc[rt][ct][v] * silu_grad(zl[r * W + j]));
                        }
                }
            }
            __syncthreads();
            store_rows(net.delta[l - 1] + (size_t)m0 * W, a0, LD, W, batch - m0, w, lane);
            bf16 *t = a0;
            a0 = a1, a1 = t;
        }
    }
}

// W^T of the hidden layers in BF16 (width x width each), 64 x 64 tiles through LDS.
__global__ void __launch_bounds__(256) transpose_bf16_kernel(const bf16 *__restrict__ w, bf16 *__restrict__ wt, int n)
{
    __shared__ bf16 t[64][66];
    const int x0 = blockIdx.x * 64, y0 = blockIdx.y * 64, c = threadIdx.x % 64;
    for (int r = threadIdx.x / 64; r < 64; r += 4)
        if (y0 + r < n && x0 + c < n)
            t[r][c] = w[(size_t)(y0 + r) * n + x0 + c];
    __syncthreads();
    for (int r = threadIdx.x / 64; r < 64; r += 4)
        if (x0 + r < n && y0 + c < n)
            wt[(size_t)(x0 + r) * n + y0 + c] = t[c][r];
}

// Weight and bias gradients of all layers: G_l[n][k] = sum_b delta_l[b][n] A_l[b][k], a 64 x 64
// tile of one layer over one slice of the batch per workgroup (40 tiles x 16 slices at width 256
// and 8,192 samples: enough to fill the device, which one workgroup per tile, 256 dependent steps
// each, did not: 2.23 ms -> 26 us).  Both operands are needed along the batch, so 64 samples at a
// time are transposed into LDS, two samples per 32-bit write.  wgrad_sum_kernel adds the slices
// in order.  Slices are the grid's fastest index: with 16 of them a slice's tiles run on one XCD
// and its operands are read into one L2.
struct WgradLayer
{
    const bf16 *delta, *act; // batch x n_out, batch x n_in (act null: the FP32 network inputs)
    int n_out, n_in, tiles_k, first_tile;
    size_t w_off, b_off;
};
struct WgradNet
{
    int n_layers, batch, rows; // rows per slice, a multiple of 64
    size_t n_params;
    const float *X;
    WgradLayer layer[kMaxFusedLayers];
};
__global__ void __launch_bounds__(256) wgrad_kernel(WgradNet net, float *__restrict__ part)
{
    constexpr int LD = 64 + 8;
    __shared__ __align__(16) bf16 As[64][LD], Bs[64][LD];
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
    const int w = tid >> 6, wm = w >> 1, wn = w & 1;
    int l = 0;
    while (l + 1 < net.n_layers && (int)blockIdx.y >= net.layer[l + 1].first_tile)
        ++l;
    const WgradLayer &ly = net.layer[l];
    const int tile = blockIdx.y - ly.first_tile, n0 = tile / ly.tiles_k * 64, k0 = tile % ly.tiles_k * 64;
    const int b0 = blockIdx.x * net.rows, b1 = min(net.batch, b0 + net.rows);
    f32x4 acc[2][2] = {};
    float db = 0.0f;
    // this thread's two samples and eight columns of a 64 x 64 block
    const int rp = 2 * (tid / 8), cg = 8 * (tid % 8);
    auto load = [&](const bf16 *src, const float *srcf, int ld, int b, int c, bf16 (&v)[8]) {
        // clamped addresses and zeroed values: no branch per element
        const int bc = min(b, b1 - 1);
        if (src && ld % 8 == 0)
        {
            const bf16x8 t = *reinterpret_cast<const bf16x8 *>(src + (size_t)bc * ld + min(c, ld - 8));
            const bool in = b < b1 && c < ld;
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[e] = in ? t[e] : (bf16)0.0f;
            return;
        }
        if (src)
        {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[e] = src[(size_t)bc * ld + min(c + e, ld - 1)];
        }
        else
        {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v[e] = (bf16)srcf[(size_t)bc * ld + min(c + e, ld - 1)];
        }
#pragma unroll
        for (int e = 0; e < 8; ++e)
            v[e] = (b < b1 && c + e < ld) ? v[e] : (bf16)0.0f;
    };
    bf16 a[2][8], x[2][8];
    auto fetch = [&](int b) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
        {
            load(ly.delta, nullptr, ly.n_out, b + rp + i, n0 + cg, a[i]);
            load(ly.act, net.X, ly.n_in, b + rp + i, k0 + cg, x[i]);
        }
    };
    fetch(b0);
    for (int b = b0; b < b1; b += 64)
    {
        if (b > b0)
            __syncthreads(); // the block before is consumed
#pragma unroll
        for (int e = 0; e < 8; ++e)
        {
            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
            *reinterpret_cast<bf16x2 *>(&As[cg + e][rp]) = bf16x2{a[0][e], a[1][e]};
            *reinterpret_cast<bf16x2 *>(&Bs[cg + e][rp]) = bf16x2{x[0][e], x[1][e]};
        }
        __syncthreads();
        if (b + 64 < b1)
            fetch(b + 64); // on its way while this block is multiplied
#pragma unroll
        for (int s = 0; s < 64; s += 32)
        {
            bf16x8 af[2], bf[2];
#pragma unroll
            for (int i = 0; i < 2; ++i)
            {
                af[i] = *reinterpret_cast<const bf16x8 *>(&As[32 * wm + 16 * i + lr][s + 8 * lk]);
                bf[i] = *reinterpret_cast<const bf16x8 *>(&Bs[32 * wn + 16 * i + lr][s + 8 * lk]);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
        }
        if (k0 == 0)
        {
            // bias: four lanes per output, 16 samples each
            float s = 0.0f;
#pragma unroll
            for (int e = 0; e < 16; ++e)
                s += (float)As[tid / 4][16 * (tid % 4) + e];
            db += s;
        }
    }
    float *out = part + (size_t)blockIdx.x * net.n_params;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v)
            {
                const int n = n0 + 32 * wm + 16 * i + 4 * lk + v, k = k0 + 32 * wn + 16 * j + lr;
                if (n < ly.n_out && k < ly.n_in)
                    out[ly.w_off + (size_t)n * ly.n_in + k] = acc[i][j][v];
            }
    if (k0 == 0)
    {
        db += __shfl_xor(db, 1);
        db += __shfl_xor(db, 2);
        const int n = n0 + tid / 4;
        if (tid % 4 == 0 && n < ly.n_out)
            out[ly.b_off + n] = db;
    }
}

// g = sum of the slices' gradients in order; the loss from the workgroups' sums of squares.
__global__ void __launch_bounds__(256) wgrad_sum_kernel(const float *__restrict__ part, int splits, size_t n,
                                                        float *__restrict__ g, const float *__restrict__ loss_part,
                                                        int n_loss, int batch, float *__restrict__ loss)
{
    const size_t i = blockIdx.x * (size_t)256 + threadIdx.x;
    if (i < n)
    {
        float s = part[i];
        for (int k = 1; k < splits; ++k)
            s += part[(size_t)k * n + i];
        g[i] = s;
    }
    if (blockIdx.x == 0)
    {
        __shared__ float red[256];
        float s = 0.0f;
        for (int k = threadIdx.x; k < n_loss; k += 256)
            s += loss_part[k];
        red[threadIdx.x] = s;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1)
        {
            if ((int)threadIdx.x < w)
                red[threadIdx.x] += red[threadIdx.x + w];
            __syncthreads();
        }
        if (threadIdx.x == 0)
            *loss = red[0] / (float)batch;
    }
}

__global__ void f32_to_bf16_kernel(const float *__restrict__ a, bf16 *__restrict__ b, long n)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256)
        b[i] = (bf16)a[i];
}

// Output layer error: d = 2 (y - t) / B (MSE), loss partials.
__global__ void __launch_bounds__(256) mse_kernel(const float *__restrict__ y, const float *__restrict__ t, int n,
                                                  bf16 *__restrict__ delta, float *__restrict__ loss)
{
    __shared__ float part[256];
    float s = 0.0f;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    {
        const float e = y[i] - t[i];
        delta[i] = (bf16)(2.0f * e / (float)n);
        s += e * e;
    }
    part[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w)
            part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        atomicAdd(loss, part[0] / (float)n);
}

// db[j] = sum_m delta[m][j]  (delta BF16, M x N)
__global__ void __launch_bounds__(256) bias_grad_kernel(const bf16 *__restrict__ delta, int M, int N,
                                                        float *__restrict__ db)
{
    const int j = blockIdx.x;
    __shared__ float part[256];
    float s = 0.0f;
    for (int m = threadIdx.x; m < M; m += 256)
        s += (float)delta[(long)m * N + j];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1)
    {
        if ((int)threadIdx.x < w)
            part[threadIdx.x] += part[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        db[j] = part[0];
}

__global__ void adam_kernel(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                            float *__restrict__ v, bf16 *__restrict__ pb, long n, float lr, float b1, float b2,
                            float eps, float c1, float c2, float wd)
{
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += (long)gridDim.x * 256)
    {
        const float gi = g[i] + wd * p[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        p[i] = pi;
        pb[i] = (bf16)pi;
    }
}

// Buffers of a batch: the hidden layers' inputs and every layer's output error.
int ensure_batch(pvl_mlp *h, int batch)
{
    if (batch <= h->cap_batch)
        return PVL_OK;
    (void)hipStreamSynchronize(stream());
    const int L = h->n_layers;
    for (int l = 1; l < L; ++l)
        (void)hipFree(h->d_act[l]), h->d_act[l] = nullptr;
    for (auto &p : h->d_delta)
        (void)hipFree(p), p = nullptr;
    (void)hipFree(h->d_loss_part);
    h->cap_batch = 0;
    h->d_loss_part = nullptr;
    for (int l = 0; l < L; ++l)
    {
        if (l > 0)
            PVL_HIP(hipMalloc(&h->d_act[l], sizeof(bf16) * (size_t)batch * h->dims[l]));
        PVL_HIP(hipMalloc(&h->d_delta[l], sizeof(bf16) * (size_t)batch * h->dims[l + 1]));
    }
    PVL_HIP(hipMalloc(&h->d_loss_part, sizeof(float) * (size_t)((batch + kRows - 1) / kRows)));
    h->cap_batch = batch;
    return PVL_OK;
}

// What the general kernels need besides: the network inputs in BF16 and the pre-activations (the fused
// pass keeps both in LDS).
int ensure_general(pvl_mlp *h, int batch)
{
    if (int st = ensure_batch(h, batch))
        return st;
    if (batch <= h->cap_general)
        return PVL_OK;
    (void)hipStreamSynchronize(stream());
    (void)hipFree(h->d_act[0]), h->d_act[0] = nullptr;
    for (auto &p : h->d_z)
        (void)hipFree(p), p = nullptr;
    h->cap_general = 0;
    PVL_HIP(hipMalloc(&h->d_act[0], sizeof(bf16) * (size_t)batch * h->dims[0]));
    for (int l = 0; l < h->n_layers; ++l)
        PVL_HIP(hipMalloc(&h->d_z[l], sizeof(float) * (size_t)batch * h->dims[l + 1]));
    h->cap_general = batch;
    return PVL_OK;
}

template <int EPI>
int launch_gemm(int M, int N, int R, const bf16 *A, long am, long ar, const bf16 *B, long bj, long br,
                const float *bias, float *outf, bf16 *outb, const float *zprev, int act)
{
    const dim3 grid((N + 63) / 64, (M + 63) / 64);
    gemm_bf16_kernel<EPI><<<grid, 256, 0, stream()>>>(M, N, R, A, am, ar, B, bj, br, bias, outf, outb, zprev, act);
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

// Forward pass storing every layer's input (BF16) and pre-activation (FP32).
int forward(pvl_mlp *h, const float *X, int batch)
{
    if (int st = ensure_general(h, batch))
        return st;
    const long nin = (long)batch * h->d_in;
    f32_to_bf16_kernel<<<256, 256, 0, stream()>>>(X, h->d_act[0], nin);
    PVL_HIP(hipGetLastError());
    const int L = h->n_layers;
    for (int l = 0; l < L; ++l)
    {
        const int K = h->dims[l], N = h->dims[l + 1];
        const bool last = l == L - 1;
        bf16 *next = last ? nullptr : h->d_act[l + 1];
        if (int st = launch_gemm<EPI_FWD>(batch, N, K, h->d_act[l], K, 1, h->d_pb + h->w_off[l], K, 1,
                                          h->d_p + h->b_off[l], h->d_z[l], next, nullptr, last ? 0 : 1))
            return st;
    }
    return PVL_OK;
}

// Backward pass of the MSE loss against T; gradients into d_g (FP32).
int backward(pvl_mlp *h, const float *T, int batch)
{
    const int L = h->n_layers;
    PVL_HIP(hipMemsetAsync(h->d_loss, 0, sizeof(float), stream()));
    // the last layer's pre-activation is the output (dims[L] == 1)
    mse_kernel<<<64, 256, 0, stream()>>>(h->d_z[L - 1], T, batch, h->d_delta[L - 1], h->d_loss);
    PVL_HIP(hipGetLastError());
    for (int l = L - 1; l >= 0; --l)
    {
        const int K = h->dims[l], N = h->dims[l + 1];
        bf16 *delta = h->d_delta[l];
        // dW_l[n][k] = sum_b delta[b][n] * A_l[b][k]
        if (int st = launch_gemm<EPI_WGRAD>(N, K, batch, delta, 1, N, h->d_act[l], 1, K, nullptr,
                                            h->d_g + h->w_off[l], nullptr, nullptr, 0))
            return st;
        bias_grad_kernel<<<N, 256, 0, stream()>>>(delta, batch, N, h->d_g + h->b_off[l]);
        PVL_HIP(hipGetLastError());
        if (l > 0)
        {
            // delta_prev[b][k] = (sum_n delta[b][n] W_l[n][k]) * SiLU'(Z_{l-1}[b][k])
            if (int st = launch_gemm<EPI_BWD>(batch, K, N, delta, N, 1, h->d_pb + h->w_off[l], 1, K, nullptr,
                                              nullptr, h->d_delta[l - 1], h->d_z[l - 1], 0))
                return st;
        }
    }
    return PVL_OK;
}

// The fused pass takes networks of up to kMaxFusedLayers layers whose activations (and, training,
// pre-activations) of kRows samples fit a workgroup's LDS: width 256 up to four layers.
constexpr size_t kFusedLds = 150 * 1024;
bool fused(const pvl_mlp *h, bool train)
{
    return h->n_layers <= kMaxFusedLayers && fused_lds_bytes(h, train) <= kFusedLds;
}

FusedNet fused_net(const pvl_mlp *h)
{
    FusedNet net{};
    net.n_layers = h->n_layers;
    for (int l = 0; l <= h->n_layers; ++l)
        net.dims[l] = h->dims[l];
    for (int l = 0; l < h->n_layers; ++l)
    {
        net.w[l] = h->d_pb + h->w_off[l];
        net.wt[l] = l >= 1 && l + 1 < h->n_layers ? h->d_pt + (size_t)(l - 1) * h->width * h->width : nullptr;
        net.bias[l] = h->d_p + h->b_off[l];
        net.act[l] = h->d_act[l];
        net.delta[l] = h->d_delta[l];
    }
    return net;
}

int fused_attributes()
{
    static bool set = false;
    if (set)
        return PVL_OK;
    PVL_HIP(hipFuncSetAttribute((const void *)fused_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)kFusedLds));
    PVL_HIP(hipFuncSetAttribute((const void *)fused_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)kFusedLds));
    set = true;
    return PVL_OK;
}

// Loss and gradients (d_loss, d_g) of a batch.
int loss_and_gradients(pvl_mlp *h, const float *X, const float *T, int batch)
{
    if (!fused(h, true))
    {
        if (int st = forward(h, X, batch))
            return st;
        return backward(h, T, batch);
    }
    if (int st = ensure_batch(h, batch))
        return st;
    if (int st = fused_attributes())
        return st;
    const int L = h->n_layers, hidden = L - 2;
    if (!h->d_part)
        PVL_HIP(hipMalloc(&h->d_part, sizeof(float) * kMaxSplits * h->n_params));
    if (hidden > 0 && !h->d_pt)
        PVL_HIP(hipMalloc(&h->d_pt, sizeof(bf16) * (size_t)hidden * h->width * h->width));
    if (!h->pt_valid)
    {
        const unsigned t = (h->width + 63) / 64;
        for (int l = 1; l <= hidden; ++l)
            transpose_bf16_kernel<<<dim3(t, t), 256, 0, stream()>>>(
                h->d_pb + h->w_off[l], h->d_pt + (size_t)(l - 1) * h->width * h->width, h->width);
        PVL_HIP(hipGetLastError());
        h->pt_valid = true;
    }
    const int groups = (batch + kRows - 1) / kRows;
    fused_kernel<true><<<groups, 64 * kFusedWaves, fused_lds_bytes(h, true), stream()>>>(fused_net(h), X, T, batch, nullptr,
                                                                             h->d_loss_part);
    PVL_HIP(hipGetLastError());
    WgradNet net{};
    net.n_layers = L, net.batch = batch, net.n_params = h->n_params, net.X = X;
    int tiles = 0;
    for (int l = 0; l < L; ++l)
    {
        WgradLayer &ly = net.layer[l];
        ly.delta = h->d_delta[l], ly.act = l ? h->d_act[l] : nullptr;
        ly.n_out = h->dims[l + 1], ly.n_in = h->dims[l];
        ly.w_off = h->w_off[l], ly.b_off = h->b_off[l];
        ly.tiles_k = (ly.n_in + 63) / 64, ly.first_tile = tiles;
        tiles += (ly.n_out + 63) / 64 * ly.tiles_k;
    }
    // slices of at least 256 samples
    const int want = std::max(1, std::min(kMaxSplits, batch / 256));
    net.rows = ((batch + want - 1) / want + 63) / 64 * 64;
    const int splits = (batch + net.rows - 1) / net.rows;
    wgrad_kernel<<<dim3(splits, tiles), 256, 0, stream()>>>(net, h->d_part);
    PVL_HIP(hipGetLastError());
    wgrad_sum_kernel<<<(unsigned)((h->n_params + 255) / 256), 256, 0, stream()>>>(
        h->d_part, splits, h->n_params, h->d_g, h->d_loss_part, groups, batch, h->d_loss);
    PVL_HIP(hipGetLastError());
    return PVL_OK;
}

} // namespace

extern "C" {

int pvl_mlp_destroy(pvl_mlp *h);

int pvl_mlp_create(pvl_mlp **out, int d_in, int width, int n_layers)
{
    PVL_API_LOCK;
    *out = nullptr;
    if (int st = ensure_init())
        return st;
    if (d_in <= 0 || width <= 0 || n_layers < 2)
    {
        set_error("mlp_create: bad sizes d_in=%d width=%d layers=%d", d_in, width, n_layers);
        return PVL_ERR_ARG;
    }
    pvl_mlp *h = new pvl_mlp;
    h->d_in = d_in;
    h->width = width;
    h->n_layers = n_layers;
    h->dims.push_back(d_in);
    for (int l = 0; l < n_layers - 1; ++l)
        h->dims.push_back(width);
    h->dims.push_back(1);
    size_t off = 0;
    for (int l = 0; l < n_layers; ++l)
    {
        h->w_off.push_back(off);
        off += (size_t)h->dims[l] * h->dims[l + 1];
        h->b_off.push_back(off);
        off += (size_t)h->dims[l + 1];
    }
    h->n_params = off;
    h->d_act.assign(n_layers, nullptr);
    h->d_z.assign(n_layers, nullptr);
    h->d_delta.assign(n_layers, nullptr);
    int st = PVL_OK;
    auto alloc = [&](void **p, size_t bytes) {
        if (!st)
            st = check_hip(hipMalloc(p, bytes), "hipMalloc(mlp)");
    };
    alloc((void **)&h->d_p, sizeof(float) * off);
    alloc((void **)&h->d_g, sizeof(float) * off);
    alloc((void **)&h->d_m, sizeof(float) * off);
    alloc((void **)&h->d_v, sizeof(float) * off);
    alloc((void **)&h->d_pb, sizeof(bf16) * off);
    alloc((void **)&h->d_loss, sizeof(float));
    if (!st)
        st = check_hip(hipMemset(h->d_m, 0, sizeof(float) * off), "hipMemset");
    if (!st)
        st = check_hip(hipMemset(h->d_v, 0, sizeof(float) * off), "hipMemset");
    if (st)
    {
        pvl_mlp_destroy(h);
        return st;
    }
    *out = h;
    return PVL_OK;
}

int pvl_mlp_destroy(pvl_mlp *h)
{
    PVL_API_LOCK;
    if (!h)
        return PVL_OK;
    (void)hipStreamSynchronize(stream());
    (void)hipFree(h->d_p);
    (void)hipFree(h->d_g);
    (void)hipFree(h->d_m);
    (void)hipFree(h->d_v);
    (void)hipFree(h->d_pb);
    (void)hipFree(h->d_loss);
    for (auto p : h->d_act)
        (void)hipFree(p);
    for (auto p : h->d_z)
        (void)hipFree(p);
    for (auto p : h->d_delta)
        (void)hipFree(p);
    (void)hipFree(h->d_part);
    (void)hipFree(h->d_loss_part);
    (void)hipFree(h->d_pt);
    delete h;
    return PVL_OK;
}

int pvl_mlp_num_params(const pvl_mlp *h, long *n)
{
    PVL_API_LOCK;
    *n = (long)h->n_params;
    return PVL_OK;
}

// Parameters (host FP32, layout: for each layer W (out x in, row-major) then b (out)).
int pvl_mlp_set_params(pvl_mlp *h, const float *params_host)
{
    PVL_API_LOCK;
    if (int st = ensure_init())
        return st;
    PVL_HIP(hipMemcpyAsync(h->d_p, params_host, sizeof(float) * h->n_params, hipMemcpyHostToDevice, stream()));
    f32_to_bf16_kernel<<<256, 256, 0, stream()>>>(h->d_p, h->d_pb, (long)h->n_params);
    PVL_HIP(hipGetLastError());
    PVL_HIP(hipMemsetAsync(h->d_m, 0, sizeof(float) * h->n_params, stream()));
    PVL_HIP(hipMemsetAsync(h->d_v, 0, sizeof(float) * h->n_params, stream()));
    PVL_HIP(hipStreamSynchronize(stream()));
    h->step = 0;
    h->pt_valid = false;
    return PVL_OK;
}

int pvl_mlp_get_params(const pvl_mlp *h, float *params_host)
{
    PVL_API_LOCK;
    PVL_HIP(hipMemcpyAsync(params_host, h->d_p, sizeof(float) * h->n_params, hipMemcpyDeviceToHost, stream()));
    PVL_HIP(hipStreamSynchronize(stream()));
    return PVL_OK;
}

// Inference: Y[b] = net(X[b, :]) for X (batch x d_in, FP32 device), Y FP32 device.
int pvl_mlp_forward(pvl_mlp *h, const float *X_dev, float *Y_dev, int batch)
{
    PVL_API_LOCK;
    if (int st = ensure_init())
        return st;
    if (batch <= 0)
        return PVL_OK;
    ProfScope prof("mlp_forward", (double)batch);
    // the fused pass's workgroups read their inputs while others write outputs: buffers that share
    // memory go through the layer buffers (inputs converted before the first output is written)
    const uintptr_t x = (uintptr_t)X_dev, y = (uintptr_t)Y_dev;
    const bool shared = x < y + sizeof(float) * (size_t)batch && y < x + sizeof(float) * (size_t)batch * h->d_in;
    if (fused(h, false) && !shared)
    {
        if (int st = fused_attributes())
            return st;
        fused_kernel<false><<<(batch + kRows - 1) / kRows, 64 * kFusedWaves, fused_lds_bytes(h, false), stream()>>>(
            fused_net(h), X_dev, nullptr, batch, Y_dev, nullptr);
        PVL_HIP(hipGetLastError());
        return PVL_OK;
    }
    if (int st = forward(h, X_dev, batch))
        return st;
    PVL_HIP(hipMemcpyAsync(Y_dev, h->d_z[h->n_layers - 1], sizeof(float) * batch, hipMemcpyDeviceToDevice,
                           stream()));
    return PVL_OK;
}

// Gradients of the mean squared error against T (no update): grads_host (n_params FP32).
int pvl_mlp_gradient(pvl_mlp *h, const float *X_dev, const float *T_dev, int batch, float *grads_host,
                     float *loss_host)
{
    PVL_API_LOCK;
    if (int st = ensure_init())
        return st;
    if (batch <= 0)
    {
        set_error("mlp_gradient: batch %d", batch);
        return PVL_ERR_ARG;
    }
    if (int st = loss_and_gradients(h, X_dev, T_dev, batch))
        return st;
    if (grads_host)
        PVL_HIP(hipMemcpyAsync(grads_host, h->d_g, sizeof(float) * h->n_params, hipMemcpyDeviceToHost, stream()));
    if (loss_host)
        PVL_HIP(hipMemcpyAsync(loss_host, h->d_loss, sizeof(float), hipMemcpyDeviceToHost, stream()));
    PVL_HIP(hipStreamSynchronize(stream()));
    return PVL_OK;
}

// One Adam step on a batch, with L2 weight decay (wd * p added to the gradient); loss_host
// (optional) receives the batch loss before the update (synchronises only if requested).
int pvl_mlp_train_step(pvl_mlp *h, const float *X_dev, const float *T_dev, int batch, float lr, float beta1,
                       float beta2, float eps, float wd, float *loss_host)
{
    PVL_API_LOCK;
    if (int st = ensure_init())
        return st;
    if (batch <= 0)
    {
        set_error("mlp_train_step: batch %d", batch);
        return PVL_ERR_ARG;
    }
    ProfScope prof("mlp_train_step", (double)batch);
    if (int st = loss_and_gradients(h, X_dev, T_dev, batch))
        return st;
    h->step += 1;
    const float c1 = 1.0f - std::pow(beta1, (float)h->step), c2 = 1.0f - std::pow(beta2, (float)h->step);
    adam_kernel<<<256, 256, 0, stream()>>>(h->d_p, h->d_g, h->d_m, h->d_v, h->d_pb, (long)h->n_params, lr, beta1,
                                           beta2, eps, c1, c2, wd);
    PVL_HIP(hipGetLastError());
    h->pt_valid = false;
    if (loss_host)
    {
        PVL_HIP(hipMemcpyAsync(loss_host, h->d_loss, sizeof(float), hipMemcpyDeviceToHost, stream()));
        PVL_HIP(hipStreamSynchronize(stream()));
    }
    return PVL_OK;
}

} // extern "C"
