// LayerNorm of the language model's layers and its adjoint (reference: language_modeling/src/utils/
// model_utils.py:52-66, cuda_fast_weight_layer.py:168-176).
//
// A lane holds four columns of every 64 (16 lanes to a row, four rows to a wave: rows of up to 256 columns, see lanes_of) or of every 256 (up to
// 1024 columns: the wave's 64 lanes): a row is read once, its mean and its variance (of the differences from the mean, as exact as
// two passes over memory) are DPP moves and, over a whole wave, row exchanges.  The adjoint forms the gradient of x in the same
// one pass and keeps the column sums for gamma and beta in registers over the rows a lane takes; the workgroups' sums are added
// up by a second, small kernel in a fixed order.
//
// Bound by HBM: 2 (forward) and 3 (adjoint) passes over rows x cols floats, 5.9 and 5.5 TB/s at 32768 x 256.  Four rows to a wave have
// four times the bytes in flight, and a sum is four moves instead of six shuffles one after the other through the LDS's crossbar; one
// wave per row, with shuffles, took 13.3 us forward and 26.0 us backward there against 11.3 and 21.9 now, 8.9 and 19.2 against 6.0 and 11.9 at 24576 x
// 128.  For the adjoint, 1024 workgroups instead of 512 took 2 us more, 256 of eight waves 0.2 us less there and 1.4 us more at 2384 rows; loads a turn ahead nothing.
#include "fwp_common.hpp"
#include "fwp_wave.hpp"

namespace fwp {
namespace {

constexpr int kWaves = 4, kBlocks = 512;

// Lanes to a row.  With 16 a wave has four rows, but few rows are few waves, the adjoint's last sums take a barrier more for each 64 columns, and what a row's
// last lanes miss of 128 or 256 columns is masked; with 64 less than a half of the lanes have columns up to 128.  16 / 64 lanes, other
// data each time: forward 800 and 2400 x 128 2.13 / 2.04, 2.24 / 2.39; 2400, 8192 and 12288 x 256 3.23 / 2.75, 4.99 / 4.71, 6.29 / 6.35, x 160 2.73 / 2.58, 4.04 / 4.03,
// 4.92 / 5.20; 100 and 8192 x 64 1.94 / 1.99, 2.54 / 3.37.  Adjoint 100, 1600 and 2400 x 128 4.98 / 4.39, 5.76 / 5.64, 5.99 / 6.37; 100, 4096, 16384 and 32768 x 256
// 6.19 / 4.46, 8.73 / 7.94, 16.9 / 15.7, 24.7 / 24.4, x 192 5.93 / 4.43, 7.98 / 7.15, 14.0 / 14.4, 20.3 / 22.4; 100 and 4096 x 64 4.37 / 4.36, 5.48 / 6.23.
int lanes_of(int rows, int cols, bool adjoint) {
    if (cols > 256) return 64;
    if (cols <= 64) return 16;
    const int few = adjoint ? (cols <= 128 ? 2000 : cols <= 192 ? 10240 : 16384) : cols <= 128 ? 1024 : 8192;
    return rows <= few ? 64 : 16;
}

// The sum over the four 16-lane rows of the wave, in all of them
__device__ __forceinline__ float rows_sum(float x) {
    float y = x;
    swap32(x, y);
    x += y, y = x;
    swap16(x, y);
    return x + y;
}

// The sum over the L lanes of a row of their sums over each 64 (L = 16) or all of their columns, in all of them: in the same order for either L, the
// columns furthest apart first, so that a row's numbers do not depend on how many rows there are.
template <int L, int V>
__device__ __forceinline__ float row_sum(const float (&y)[V]) {
    float x = y[0];
    if constexpr (L == 64) {
#pragma unroll
        for (int i = 1; i < V; i++) x += y[i];
        x = rows_sum(x);
    } else if constexpr (V == 4) x = (y[0] + y[2]) + (y[1] + y[3]);
    else if constexpr (V == 2) x = y[0] + y[1];
    x += dpp<kRowRor8>(x);
    x += dpp<kRowRor4>(x);          // the halves are alike by now
    x += dpp<kQuadXor2>(x);
    x += dpp<kQuadXor1>(x);
    return x;
}

__device__ __forceinline__ float4 load4(const float *p, bool ok) {
    return ok ? *reinterpret_cast<const float4 *>(p) : make_float4(0.f, 0.f, 0.f, 0.f);
}

template <int L, int V>
__global__ __launch_bounds__(64 * kWaves) void k_norm_fwd(const float *__restrict__ x, const float *__restrict__ gamma,
                                                          const float *__restrict__ beta, float *__restrict__ y,
                                                          float *__restrict__ stats, int rows, int cols, float eps) {
    const int lane = threadIdx.x % L, row = blockIdx.x * (64 * kWaves / L) + threadIdx.x / L;
    if (row >= rows) return;        // all lanes of a row together
    const float *src = x + (int64_t)row * cols;
    float4 v[V];
    float s[V];
#pragma unroll
    for (int i = 0; i < V; i++) {
        const int c = 4 * (lane + L * i);
        v[i] = load4(src + c, c < cols);
    }
#pragma unroll
    for (int i = 0; i < V; i++) s[i] = (v[i].x + v[i].y) + (v[i].z + v[i].w);
    const float mean = row_sum<L>(s) / cols;
#pragma unroll
    for (int i = 0; i < V; i++) {
        const float a = v[i].x - mean, b = v[i].y - mean, c = v[i].z - mean, d = v[i].w - mean;
        s[i] = 4 * (lane + L * i) < cols ? fmaf(a, a, b * b) + fmaf(c, c, d * d) : 0.f;
    }
    const float rstd = 1.f / sqrtf(row_sum<L>(s) / cols + eps);
#pragma unroll
    for (int i = 0; i < V; i++) {
        const int c = 4 * (lane + L * i);
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
template <int L, int V>
__global__ __launch_bounds__(64 * kWaves) void k_norm_bwd(const float *__restrict__ gy, const float *__restrict__ x,
                                                          const float *__restrict__ stats, const float *__restrict__ gamma,
                                                          float *__restrict__ gx,
                                                          float *__restrict__ part, int rows, int cols) {
#pragma clang fp contract(off)      // the same fused operations for any L and V, and so the same numbers
    constexpr int R = 64 * kWaves / L;      // rows of a workgroup at once
    const int lane = threadIdx.x % L, wave = threadIdx.x / 64;
    float4 gam[V], sg[V], sb[V];
#pragma unroll
    for (int i = 0; i < V; i++) {
        const int c = 4 * (lane + L * i);
        gam[i] = load4(gamma + c, c < cols);
        sg[i] = sb[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    for (int64_t row = (int64_t)blockIdx.x * R + threadIdx.x / L; row < rows; row += (int64_t)gridDim.x * R) {
        const int64_t at = row * cols;
        const float2 st = *reinterpret_cast<const float2 *>(stats + 2 * row);
        float4 g[V], xh[V];
        float sums[V], products[V];
#pragma unroll
        for (int i = 0; i < V; i++) {
            const int c = 4 * (lane + L * i);
            g[i] = load4(gy + at + c, c < cols), xh[i] = load4(x + at + c, c < cols);
        }
#pragma unroll
        for (int i = 0; i < V; i++) {
            const float4 d = g[i], w = xh[i];
            xh[i] = make_float4((w.x - st.x) * st.y, (w.y - st.x) * st.y, (w.z - st.x) * st.y, (w.w - st.x) * st.y);
            sb[i].x += d.x, sb[i].y += d.y, sb[i].z += d.z, sb[i].w += d.w;
            sg[i] = make_float4(fmaf(d.x, xh[i].x, sg[i].x), fmaf(d.y, xh[i].y, sg[i].y), fmaf(d.z, xh[i].z, sg[i].z), fmaf(d.w, xh[i].w, sg[i].w));
            g[i] = make_float4(d.x * gam[i].x, d.y * gam[i].y, d.z * gam[i].z, d.w * gam[i].w);
            sums[i] = (g[i].x + g[i].y) + (g[i].z + g[i].w);
            products[i] = fmaf(g[i].x, xh[i].x, g[i].y * xh[i].y) + fmaf(g[i].z, xh[i].z, g[i].w * xh[i].w);
        }
        const float s = row_sum<L>(sums) / cols, t = row_sum<L>(products) / cols;
#pragma unroll
        for (int i = 0; i < V; i++) {
            const int c = 4 * (lane + L * i);
            if (c >= cols) continue;
            float4 o = make_float4(st.y * fmaf(-xh[i].x, t, g[i].x - s), st.y * fmaf(-xh[i].y, t, g[i].y - s),
                                   st.y * fmaf(-xh[i].z, t, g[i].z - s), st.y * fmaf(-xh[i].w, t, g[i].w - s));
            *reinterpret_cast<float4 *>(gx + at + c) = o;
        }
    }
    // this workgroup's column sums: [gamma | beta][cols]
    __shared__ float4 sh[kWaves][L];
#pragma unroll
    for (int i = 0; i < V; i++)
#pragma unroll
        for (int w = 0; w < 2; w++) {
            float4 o = w ? sb[i] : sg[i];
            if constexpr (L == 16) o = make_float4(rows_sum(o.x), rows_sum(o.y), rows_sum(o.z), rows_sum(o.w));
            __syncthreads();
            if (threadIdx.x % 64 < L) sh[wave][lane] = o;
            __syncthreads();
            const int c = 4 * (lane + L * i);
            if (threadIdx.x >= L || c >= cols) continue;
            o = sh[0][lane];
#pragma unroll
            for (int k = 1; k < kWaves; k++) o.x += sh[k][lane].x, o.y += sh[k][lane].y, o.z += sh[k][lane].z, o.w += sh[k][lane].w;
            *reinterpret_cast<float4 *>(part + ((int64_t)blockIdx.x * 2 + w) * cols + c) = o;
        }
}

// ggamma, gbeta = the workgroups' sums added up: 16 columns x 64 slices of the workgroups per workgroup, a slice's loads all at once, for up to 64, 256 or 512
// workgroups (eight loads for few of them took 0.2 us more, a branch in the kernel 0.2 us more for many)
constexpr int kSlices = 64;
template <int EACH>
__global__ __launch_bounds__(1024) void k_norm_params(const float *__restrict__ part, float *__restrict__ ggamma,
                                                      float *__restrict__ gbeta, int blocks, int cols) {
    __shared__ float sh[16][16];
    const int c = threadIdx.x % 16, q = threadIdx.x / 16, col = blockIdx.x * 16 + c;
    const float *const from = part + min(col, 2 * cols - 1);
    float x[EACH], s = 0.f;
#pragma unroll
    for (int i = 0; i < EACH; i++) x[i] = from[(int64_t)min(q + kSlices * i, blocks - 1) * 2 * cols];
#pragma unroll
    for (int i = 0; i < EACH; i++) s += q + kSlices * i < blocks ? x[i] : 0.f;
    s = rows_sum(s);
    if (q % 4 == 0) sh[q / 4][c] = s;
    __syncthreads();
    if (q || col >= 2 * cols) return;
    float t[4] = {};
#pragma unroll
    for (int k = 0; k < 16; k++) t[k % 4] += sh[k][c];
    s = (t[0] + t[1]) + (t[2] + t[3]);
    (col < cols ? ggamma : gbeta)[col < cols ? col : col - cols] = s;
}

int blocks_of(int rows, int cols) {
    const int at_once = 64 * kWaves / lanes_of(rows, cols, true);
    return (int)std::min<int64_t>(((int64_t)rows + at_once - 1) / at_once, kBlocks);
}

}  // namespace

bool layer_norm_supported(int cols) { return cols >= 4 && cols <= 1024 && cols % 4 == 0; }
int64_t layer_norm_workspace(int rows, int cols) { return (int64_t)blocks_of(rows, cols) * 2 * cols; }

#define FWP_BY_COLS(LANES, LAUNCH)                                                                                           \
    if (cols <= 256 && LANES == 64) LAUNCH(64, 1);                                                                           \
    else if (cols <= 64) LAUNCH(16, 1);                                                                                      \
    else if (cols <= 128) LAUNCH(16, 2);                                                                                     \
    else if (cols <= 256) LAUNCH(16, 4);                                                                                     \
    else if (cols <= 512) LAUNCH(64, 2);                                                                                     \
    else LAUNCH(64, 4)

int layer_norm_fwd(const float *x, const float *gamma, const float *beta, float *y, float *stats, int rows, int cols,
                   float eps, hipStream_t s) {
    const int lanes = lanes_of(rows, cols, false), at_once = 64 * kWaves / lanes;
    const dim3 grid((unsigned)(((int64_t)rows + at_once - 1) / at_once)), block(64 * kWaves);
#define FWP_FWD(L, V) hipLaunchKernelGGL((k_norm_fwd<L, V>), grid, block, 0, s, x, gamma, beta, y, stats, rows, cols, eps)
    FWP_BY_COLS(lanes, FWP_FWD);
#undef FWP_FWD
    return (int)hipGetLastError();
}

int layer_norm_bwd(const float *gy, const float *x, const float *stats, const float *gamma, float *gx,
                   float *ggamma, float *gbeta, float *workspace, int rows, int cols, hipStream_t s) {
    const int blocks = blocks_of(rows, cols), lanes = lanes_of(rows, cols, true);
    const dim3 grid(blocks), block(64 * kWaves);
#define FWP_BWD(L, V) hipLaunchKernelGGL((k_norm_bwd<L, V>), grid, block, 0, s, gy, x, stats, gamma, gx, workspace, rows, cols)
    FWP_BY_COLS(lanes, FWP_BWD);
#undef FWP_BWD
    const auto sum = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((2 * cols + 15) / 16), dim3(1024), 0, s, workspace, ggamma, gbeta, blocks, cols); };
    if (blocks <= kSlices) sum(k_norm_params<1>);
    else if (blocks <= 4 * kSlices) sum(k_norm_params<4>);
    else sum(k_norm_params<kBlocks / kSlices>);
    return (int)hipGetLastError();
}
#undef FWP_BY_COLS

}  // namespace fwp
