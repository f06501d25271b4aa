// Training and batch inference of the stencil-weight MLP on the gfx950 matrix cores.
//
// A batch is at most a few thousand rows of a 128-256-256-256-32 network: about 1 GFLOP
// forward, a few microseconds at the matrix rate, so what bounds a pass is the chain of
// dependent launches and memory round trips. It runs in three launches:
//   k_mlp_prep   zeroes the gradients and the loss and transposes the weights that the
//                backward products need with the other index contiguous;
//   k_mlp        one workgroup carries 16 (or 32) rows of the batch through all four
//                layers, the loss and back: the activations pass between layers in LDS, the
//                pre-activations that GELU' needs stay in registers (the wavefront that
//                computes a column forward is the one that needs it backward), the
//                weights stream from L2 as matrix fragments;
//   k_mlp_wgrad  the weight gradients dZ^T H of all layers, 64x64 tiles over slices of the
//                batch, with the bias gradients summed while the tiles are staged.
// Against one launch per product, loss and column sum (18 launches, the operands of the
// transposed products read two bytes at a time): 4096 rows forward and back
// 1358 -> 83 us a pass (of it k_mlp 33, k_mlp_wgrad 28, k_mlp_prep 4).
//
// BF16 operands, FP32 accumulation; the activations and the dZ are rounded to BF16
// where they become operands, as the weights' copy is.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mlp.h"

namespace rbfx {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kHidLds = kHid + 8;  // LDS row stride: 16-byte aligned rows, 4 banks apart
constexpr int kWgTile = 64, kWgRows = 128, kWgSlice = 256;  // weight gradient: tile, staged rows, batch slice

// ---------------------------------------------------------------- prepare
__global__ __launch_bounds__(256) void k_mlp_prep(MlpPass a)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (a.target) {
        if (i < mlp_n_params()) a.grads[i] = 0.f;
        if (i == 0) *a.loss = 0.f;
    }
    if (i >= mlp_n_wbf16()) return;
    const __bf16 w = a.w[i];
    if (a.wcopy) a.wcopy[i] = w;  // (weights that are not 16-byte aligned)
    if (!a.target) return;
    int l = 0;
    while (l + 1 < kMlpLayers && i >= mlp_wb_off(l + 1)) ++l;
    if (l == 0) return;  // (no gradient passes through the inputs)
    const int64_t r = i - mlp_wb_off(l);
    const int n = (int)(r / kHid), k = (int)(r % kHid);
    a.wt[mlp_wb_off(l) - mlp_wb_off(1) + (int64_t)k * mlp_n(l) + n] = w;
}

// ---------------------------------------------------------------- forward and back
// acc[i][j] += A (rows 16 i of the LDS buffer) B^T (columns n0 + 16 j of W), reduction K
template <int MT, int NT, int K>
__device__ __forceinline__ void mlp_product(const __bf16* act, const __bf16* __restrict__ W, int n0, int lane,
                                            f32x4 (&acc)[MT][NT])
{
    constexpr int KS = K / 32;
    const int fr = lane & 15, fk = (lane >> 4) * 8;
    bf16x8 b[KS][NT];  // the whole panel in flight at once: one L2 round trip per layer
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < NT; ++j)
            b[s][j] = *reinterpret_cast<const bf16x8*>(W + (int64_t)(n0 + 16 * j + fr) * K + 32 * s + fk);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            const bf16x8 av = *reinterpret_cast<const bf16x8*>(act + (16 * i + fr) * kHidLds + 32 * s + fk);
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, b[s][j], acc[i][j], 0, 0, 0);
        }
}

// rows of the LDS buffer to the workspace (16 bytes per thread, whole rows of kHid)
template <int MT>
__device__ __forceinline__ void mlp_store(const __bf16* act, __bf16* out, int64_t m0, int M)
{
#pragma unroll
    for (int q = 0; q < MT * 2; ++q) {
        const int c = q * 256 + threadIdx.x, r = c >> 5, col = (c & 31) * 8;
        if (m0 + r < M)
            *reinterpret_cast<bf16x8*>(out + (m0 + r) * kHid + col) =
                *reinterpret_cast<const bf16x8*>(act + r * kHidLds + col);
    }
}

// MT: 16-row tiles of the batch per workgroup. Four wavefronts, 64 hidden columns each.
template <int MT, bool TRAIN>
__global__ __launch_bounds__(256) void k_mlp(MlpPass a)
{
    __shared__ __attribute__((aligned(16))) __bf16 act[2][MT * 16 * kHidLds];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int64_t m0 = (int64_t)blockIdx.x * (MT * 16);
    const int col = lane & 15, row = (lane >> 4) * 4;  // D layout: column lane % 16, rows row + q
    const __bf16* W = a.wcopy ? a.wcopy : a.w;

    // inputs (rows past the batch are zero)
#pragma unroll
    for (int q = 0; q < MT; ++q) {
        const int c = q * 256 + t, r = c >> 4, k = (c & 15) * 8;
        bf16x8 v = {};
        if (m0 + r < a.M) {
            const __bf16* x = a.x + (m0 + r) * kInPad + k;
            if (!a.xcopy) {
                v = *reinterpret_cast<const bf16x8*>(x);
            } else {  // (inputs that are not 16-byte aligned)
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = x[i];
                if (TRAIN) *reinterpret_cast<bf16x8*>(a.xcopy + (m0 + r) * kInPad + k) = v;
            }
        }
        *reinterpret_cast<bf16x8*>(&act[0][r * kHidLds + k]) = v;
    }
    __syncthreads();

    f32x4 Z[kMlpLayers - 1][MT][4];
#pragma unroll
    for (int l = 0; l < kMlpLayers - 1; ++l) {
        f32x4 acc[MT][4];
        if (l == 0) mlp_product<MT, 4, kInPad>(act[0], W + mlp_wb_off(0), 64 * w, lane, acc);
        else mlp_product<MT, 4, kHid>(act[l & 1], W + mlp_wb_off(l), 64 * w, lane, acc);
        __bf16* out = act[(l + 1) & 1];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = 64 * w + 16 * j + col;
            const float bias = a.params[mlp_b_off(l) + n];
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float z = acc[i][j][q] + bias;
                    Z[l][i][j][q] = z;
                    out[(16 * i + row + q) * kHidLds + n] = (__bf16)gelu_tanh(z);
                }
        }
        __syncthreads();
        if (TRAIN) mlp_store<MT>(out, a.H[l], m0, a.M);
    }

    // outputs (32 columns: the first two wavefronts), loss and its gradient
    float part = 0.f;
    if (w < 2) {
        f32x4 acc[MT][1];
        mlp_product<MT, 1, kHid>(act[1], W + mlp_wb_off(3), 16 * w, lane, acc);
        const int n = 16 * w + col;
        const float bias = a.params[mlp_b_off(3) + n];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = 16 * i + row + q;
                const int64_t m = m0 + r;
                const float y = acc[i][0][q] + bias;
                if (a.y && m < a.M) a.y[m * kOutPad + n] = y;
                if (TRAIN) {
                    float d = 0.f, wm = 1.f;
                    if (m < a.M && n < a.n_out) {
                        wm = a.row_weight ? a.row_weight[m] : 1.0f;
                        d = y - a.target[m * a.n_out + n];
                        part += wm * d * d;
                    }
                    const __bf16 g = (__bf16)(2.0f * wm * d / ((float)a.M * (float)a.n_out));
                    act[0][r * kHidLds + n] = g;
                    if (m < a.M) a.dY[m * kOutPad + n] = g;
                }
            }
    }
    if (!TRAIN) return;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) part += __shfl_xor(part, s, 64);
    if (w < 2 && lane == 0) atomicAdd(a.loss, part / ((float)a.M * (float)a.n_out));
    __syncthreads();

#pragma unroll
    for (int l = kMlpLayers - 1; l >= 1; --l) {
        f32x4 acc[MT][4];
        const __bf16* Wt = a.wt + mlp_wb_off(l) - mlp_wb_off(1);
        const __bf16* in = act[(l + 1) & 1];  // dY in buffer 0, then 1, 0
        if (l == kMlpLayers - 1) mlp_product<MT, 4, kOutPad>(in, Wt, 64 * w, lane, acc);
        else mlp_product<MT, 4, kHid>(in, Wt, 64 * w, lane, acc);
        __bf16* out = act[l & 1];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    out[(16 * i + row + q) * kHidLds + 64 * w + 16 * j + col] =
                        (__bf16)(acc[i][j][q] * gelu_tanh_grad(Z[l - 1][i][j][q]));
        __syncthreads();
        mlp_store<MT>(out, a.dZ[l - 1], m0, a.M);
    }
}

// ---------------------------------------------------------------- weight gradients
// One 64x64 tile of dZ_l^T H_(l-1) over a slice of the batch, added to the gradients. Both
// operands lie with the batch index outermost, so a thread reads 16 bytes (8 columns) of
// two rows and writes them to LDS as 8 pairs, the batch index contiguous there.
__device__ __forceinline__ void wg_stage(const __bf16* src, int64_t ld, int n_cols, int64_t m0, int64_t m_end,
                                         __bf16 (*dst)[kWgRows + 8], float (&colsum)[8])
{
    const int cb = (threadIdx.x & 7) * 8, rp = threadIdx.x >> 3;
#pragma unroll
    for (int h = 0; h < kWgRows / 64; ++h) {
        const int r = 64 * h + 2 * rp;
        bf16x8 u = {}, v = {};
        if (cb < n_cols) {
            if (m0 + r < m_end) u = *reinterpret_cast<const bf16x8*>(src + (m0 + r) * ld + cb);
            if (m0 + r + 1 < m_end) v = *reinterpret_cast<const bf16x8*>(src + (m0 + r + 1) * ld + cb);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            *reinterpret_cast<bf16x2*>(&dst[cb + i][r]) = bf16x2{u[i], v[i]};
            colsum[i] += (float)u[i] + (float)v[i];
        }
    }
}

__global__ __launch_bounds__(256) void k_mlp_wgrad(MlpPass a)
{
    __shared__ __attribute__((aligned(16))) __bf16 As[kWgTile][kWgRows + 8], Bs[kWgTile][kWgRows + 8];
    // tile list: layer 0 4x2, layers 1 and 2 4x4, layer 3 1x4
    int id = blockIdx.x, l = 0;
    if (id >= 40) {
        l = 3;
        id -= 40;
    } else if (id >= 24) {
        l = 2;
        id -= 24;
    } else if (id >= 8) {
        l = 1;
        id -= 8;
    }
    const int N = mlp_n(l), K = mlp_k(l), kt = K / kWgTile;
    const int n0 = (id / kt) * kWgTile, k0 = (id % kt) * kWgTile;
    // (selected, not indexed: an indexed kernel argument would be copied to scratch memory)
    const __bf16* dZ = (l == 3 ? a.dY : (l == 2 ? a.dZ[2] : (l == 1 ? a.dZ[1] : a.dZ[0]))) + n0;
    const __bf16* Hin = (l == 3 ? a.H[2] : (l == 2 ? a.H[1] : (l == 1 ? a.H[0] : (a.xcopy ? a.xcopy : a.x)))) + k0;
    const int64_t mb = (int64_t)blockIdx.y * kWgSlice;
    const int64_t me = mb + kWgSlice < a.M ? mb + kWgSlice : a.M;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
    const int fr = lane & 15, fk = (lane >> 4) * 8;
    float cs[8] = {}, unused[8] = {};
    f32x4 acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int64_t m = mb; m < me; m += kWgRows) {
        wg_stage(dZ, N, N - n0, m, me, As, cs);
        wg_stage(Hin, K, K - k0, m, me, Bs, unused);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < kWgRows / 32; ++s) {
            bf16x8 x[2], y[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) x[i] = *reinterpret_cast<const bf16x8*>(&As[wm + 16 * i + fr][32 * s + fk]);
#pragma unroll
            for (int j = 0; j < 2; ++j) y[j] = *reinterpret_cast<const bf16x8*>(&Bs[wn + 16 * j + fr][32 * s + fk]);
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[i], y[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = n0 + wm + 16 * i + (lane >> 4) * 4 + q, k = k0 + wn + 16 * j + fr;
                if (n < N) atomicAdd(&a.grads[mlp_w_off(l) + (int64_t)n * K + k], acc[i][j][q]);
            }
    if (k0 == 0) {  // bias: the 32 threads of one column block
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            float v = cs[i];
            v += __shfl_xor(v, 8, 64);
            v += __shfl_xor(v, 16, 64);
            v += __shfl_xor(v, 32, 64);
            const int n = n0 + (t & 7) * 8 + i;
            if (lane < 8 && n < N) atomicAdd(&a.grads[mlp_b_off(l) + n], v);
        }
    }
}

// One pass. 16 rows per workgroup fill the chip at the training batch (4096 rows, 256
// workgroups); beyond 8192 rows 32 per workgroup halve the weights read from L2 per row.
hipError_t launch_mlp(const MlpPass& a, hipStream_t s)
{
    if (a.M <= 0) return hipSuccess;
    if (a.target || a.wcopy)
        hipLaunchKernelGGL(k_mlp_prep, dim3((unsigned)((mlp_n_params() + 255) / 256)), dim3(256), 0, s, a);
    const int rows = a.M <= 8192 ? 16 : 32;
    const dim3 grid((unsigned)((a.M + rows - 1) / rows));
    if (a.target) {
        if (rows == 16) hipLaunchKernelGGL((k_mlp<1, true>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((k_mlp<2, true>), grid, dim3(256), 0, s, a);
        hipLaunchKernelGGL(k_mlp_wgrad, dim3(44, (unsigned)((a.M + kWgSlice - 1) / kWgSlice)), dim3(256), 0, s, a);
    } else {
        if (rows == 16) hipLaunchKernelGGL((k_mlp<1, false>), grid, dim3(256), 0, s, a);
        else hipLaunchKernelGGL((k_mlp<2, false>), grid, dim3(256), 0, s, a);
    }
    return hipGetLastError();
}

// Adam (Kingma & Ba 2015) with bias correction
__global__ __launch_bounds__(256) void k_adam(int64_t n, float* p, const float* g, float* m, float* v, float lr,
                                              float b1, float b2, float eps, float c1, float c2)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

hipError_t launch_adam(int64_t n, float* p, const float* g, float* m, float* v, float lr, float b1, float b2,
                       float eps, int t, hipStream_t s)
{
    const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
    hipLaunchKernelGGL(k_adam, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, p, g, m, v, lr, b1, b2, eps, c1,
                       c2);
    return hipGetLastError();
}

// BF16 copy of the Wt blocks of the flat FP32 parameter array
__global__ __launch_bounds__(256) void k_params_to_bf16(const float* p, __bf16* wb)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= mlp_n_wbf16()) return;
    int l = 0;
    while (l + 1 < kMlpLayers && i >= mlp_wb_off(l + 1)) ++l;
    wb[i] = (__bf16)p[mlp_w_off(l) + (i - mlp_wb_off(l))];
}

hipError_t launch_params_to_bf16(const float* p, __bf16* wb, hipStream_t s)
{
    hipLaunchKernelGGL(k_params_to_bf16, dim3((unsigned)((mlp_n_wbf16() + 255) / 256)), dim3(256), 0, s, p, wb);
    return hipGetLastError();
}

}  // namespace rbfx
