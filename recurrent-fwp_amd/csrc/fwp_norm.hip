// LayerNorm of the language model's layers and its adjoint (reference: language_modeling/src/utils/
// model_utils.py:52-66, cuda_fast_weight_layer.py:168-176).
//
// One wave per row, a float4 of the row per lane and 256 columns (up to four of them): a row is read once, its mean
// and its variance (of the differences from the mean, as exact as two passes over memory) are butterflies
// inside the wave.  The adjoint forms the gradient of x in the same one pass and keeps the column sums for gamma and
// beta in registers over the rows a wave takes; the workgroups' sums are added up by a second, small kernel in
// a fixed order.  Bound by HBM: 2 (forward) and 3 (adjoint) passes over rows x cols floats.
#include "fwp_common.hpp"

namespace fwp {
namespace {

constexpr int kWaves = 4, kBlocks = 512;

__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) x += __shfl_xor(x, m, 64);
    return x;
}

__device__ __forceinline__ float4 load4(const float *p, bool ok) {
    return ok ? *reinterpret_cast<const float4 *>(p) : make_float4(0.f, 0.f, 0.f, 0.f);
}

template <int V>
__global__ __launch_bounds__(64 * kWaves) void k_norm_fwd(const float *__restrict__ x, const float *__restrict__ gamma,
                                                          const float *__restrict__ beta, float *__restrict__ y,
                                                          float *__restrict__ stats, int rows, int cols, float eps) {
    const int lane = threadIdx.x % 64, row = blockIdx.x * kWaves + threadIdx.x / 64;
    if (row >= rows) return;
    const float *src = x + (int64_t)row * cols;
    float4 v[V];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < V; i++) {
        const int c = 4 * (lane + 64 * i);
        v[i] = load4(src + c, c < cols);
        s += (v[i].x + v[i].y) + (v[i].z + v[i].w);
    }
    const float mean = wave_sum(s) / cols;
    s = 0.f;
#pragma unroll
    for (int i = 0; i < V; i++)
        if (4 * (lane + 64 * i) < cols) {
            const float a = v[i].x - mean, b = v[i].y - mean, c = v[i].z - mean, d = v[i].w - mean;
            s += (a * a + b * b) + (c * c + d * d);
        }
    const float rstd = 1.f / sqrtf(wave_sum(s) / cols + eps);
#pragma unroll
    for (int i = 0; i < V; i++) {
        const int c = 4 * (lane + 64 * i);
        if (c >= cols) continue;
        const float4 g = load4(gamma + c, true), b = load4(beta + c, true);
        float4 o;
        o.x = (v[i].x - mean) * rstd * g.x + b.x, o.y = (v[i].y - mean) * rstd * g.y + b.y;
        o.z = (v[i].z - mean) * rstd * g.z + b.z, o.w = (v[i].w - mean) * rstd * g.w + b.w;
        *reinterpret_cast<float4 *>(y + (int64_t)row * cols + c) = o;
    }
    if (stats && lane == 0) *reinterpret_cast<float2 *>(stats + 2 * (int64_t)row) = make_float2(mean, rstd);
}

// gx = rstd (g - mean(g) - xh mean(g xh)),  g = gy gamma, xh = (x - mean) rstd
template <int V>
__global__ __launch_bounds__(64 * kWaves) void k_norm_bwd(const float *__restrict__ gy, const float *__restrict__ x,
                                                          const float *__restrict__ stats, const float *__restrict__ gamma,
                                                          float *__restrict__ gx,
                                                          float *__restrict__ part, int rows, int cols) {
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    float4 gam[V], sg[V], sb[V];
#pragma unroll
    for (int i = 0; i < V; i++) {
        const int c = 4 * (lane + 64 * i);
        gam[i] = load4(gamma + c, c < cols);
        sg[i] = sb[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    for (int row = blockIdx.x * kWaves + wave; row < rows; row += gridDim.x * kWaves) {
        const int64_t at = (int64_t)row * cols;
        const float2 st = *reinterpret_cast<const float2 *>(stats + 2 * (int64_t)row);
        float4 g[V], xh[V];
        float s = 0.f, t = 0.f;
#pragma unroll
        for (int i = 0; i < V; i++) {
            const int c = 4 * (lane + 64 * i);
            const float4 d = load4(gy + at + c, c < cols), w = load4(x + at + c, c < cols);
            xh[i] = make_float4((w.x - st.x) * st.y, (w.y - st.x) * st.y, (w.z - st.x) * st.y, (w.w - st.x) * st.y);
            sb[i].x += d.x, sb[i].y += d.y, sb[i].z += d.z, sb[i].w += d.w;
            sg[i].x += d.x * xh[i].x, sg[i].y += d.y * xh[i].y, sg[i].z += d.z * xh[i].z, sg[i].w += d.w * xh[i].w;
            g[i] = make_float4(d.x * gam[i].x, d.y * gam[i].y, d.z * gam[i].z, d.w * gam[i].w);
            s += (g[i].x + g[i].y) + (g[i].z + g[i].w);
            t += (g[i].x * xh[i].x + g[i].y * xh[i].y) + (g[i].z * xh[i].z + g[i].w * xh[i].w);
        }
        s = wave_sum(s) / cols;
        t = wave_sum(t) / cols;
#pragma unroll
        for (int i = 0; i < V; i++) {
            const int c = 4 * (lane + 64 * i);
            if (c >= cols) continue;
            float4 o = make_float4(st.y * (g[i].x - s - xh[i].x * t), st.y * (g[i].y - s - xh[i].y * t),
                                   st.y * (g[i].z - s - xh[i].z * t), st.y * (g[i].w - s - xh[i].w * t));
            *reinterpret_cast<float4 *>(gx + at + c) = o;
        }
    }
    // this workgroup's column sums: [gamma | beta][cols]
    __shared__ float4 sh[kWaves][64];
#pragma unroll
    for (int i = 0; i < V; i++)
        for (int w = 0; w < 2; w++) {
            __syncthreads();
            sh[wave][lane] = w ? sb[i] : sg[i];
            __syncthreads();
            const int c = 4 * (lane + 64 * i);
            if (wave || c >= cols) continue;
            float4 o = sh[0][lane];
#pragma unroll
            for (int k = 1; k < kWaves; k++) o.x += sh[k][lane].x, o.y += sh[k][lane].y, o.z += sh[k][lane].z, o.w += sh[k][lane].w;
            *reinterpret_cast<float4 *>(part + ((int64_t)blockIdx.x * 2 + w) * cols + c) = o;
        }
}

// ggamma, gbeta = the workgroups' sums added up: 16 columns x 16 slices of the workgroups per workgroup
__global__ __launch_bounds__(256) void k_norm_params(const float *__restrict__ part, float *__restrict__ ggamma,
                                                     float *__restrict__ gbeta, int blocks, int cols) {
    __shared__ float sh[16][17];
    const int c = threadIdx.x % 16, q = threadIdx.x / 16, col = blockIdx.x * 16 + c;
    float s = 0.f;
    if (col < 2 * cols) {
#pragma unroll 8
        for (int b = q; b < blocks; b += 16) s += part[(int64_t)b * 2 * cols + col];
    }
    sh[q][c] = s;
    __syncthreads();
    if (q || col >= 2 * cols) return;
    for (int k = 1; k < 16; k++) s += sh[k][c];
    (col < cols ? ggamma : gbeta)[col < cols ? col : col - cols] = s;
}

int blocks_of(int rows) { return rows < kBlocks * kWaves ? (rows + kWaves - 1) / kWaves : kBlocks; }

}  // namespace

bool layer_norm_supported(int cols) { return cols >= 4 && cols <= 1024 && cols % 4 == 0; }
int64_t layer_norm_workspace(int rows, int cols) { return (int64_t)blocks_of(rows) * 2 * cols; }

int layer_norm_fwd(const float *x, const float *gamma, const float *beta, float *y, float *stats, int rows, int cols,
                   float eps, hipStream_t s) {
    const dim3 grid((rows + kWaves - 1) / kWaves), block(64 * kWaves);
    const int v = (cols + 255) / 256;
    if (v == 1) hipLaunchKernelGGL(k_norm_fwd<1>, grid, block, 0, s, x, gamma, beta, y, stats, rows, cols, eps);
    else if (v == 2) hipLaunchKernelGGL(k_norm_fwd<2>, grid, block, 0, s, x, gamma, beta, y, stats, rows, cols, eps);
    else hipLaunchKernelGGL(k_norm_fwd<4>, grid, block, 0, s, x, gamma, beta, y, stats, rows, cols, eps);
    return (int)hipGetLastError();
}

int layer_norm_bwd(const float *gy, const float *x, const float *stats, const float *gamma, float *gx,
                   float *ggamma, float *gbeta, float *workspace, int rows, int cols, hipStream_t s) {
    const int blocks = blocks_of(rows), v = (cols + 255) / 256;
    const dim3 grid(blocks), block(64 * kWaves);
    if (v == 1) hipLaunchKernelGGL(k_norm_bwd<1>, grid, block, 0, s, gy, x, stats, gamma, gx, workspace, rows, cols);
    else if (v == 2) hipLaunchKernelGGL(k_norm_bwd<2>, grid, block, 0, s, gy, x, stats, gamma, gx, workspace, rows, cols);
    else hipLaunchKernelGGL(k_norm_bwd<4>, grid, block, 0, s, gy, x, stats, gamma, gx, workspace, rows, cols);
    hipLaunchKernelGGL(k_norm_params, dim3((2 * cols + 15) / 16), dim3(256), 0, s, workspace, ggamma, gbeta, blocks, cols);
    return (int)hipGetLastError();
}

}  // namespace fwp
