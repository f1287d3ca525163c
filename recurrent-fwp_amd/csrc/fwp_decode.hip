// One token per sequence through the Delta-Net language model (decoding; up to 64 sequences): products of a few rows
// with the weights, the delta rule's single step from the layer's projection, and the embedding.
//
// Nothing here is large: a layer's weights are 3 MB, which the chip reads in under a microsecond, and its rows fit one
// MFMA tile.  What counts is the number of launches and the latency of each, so a layer is five kernels:
// projection, step, output projection, and the two feed-forward products, with LayerNorm, biases, ReLU and
// residuals inside them.  (Decoding 8 sequences with d_model 256, 16 layers: 82 launches of 3-5 us where the layers'
// general path takes 180.)
#include "fwp_common.hpp"
#include "fwp_wave.hpp"

namespace fwp {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4f ld4(const float *p) { return *reinterpret_cast<const v4f *>(p); }

struct RowsArgs {
    const float *x, *gamma, *beta;      // rows [rows,K]; LayerNorm on the way in (LN)
    float eps;
    float *y;                           // the normalised rows, or NULL
    const float *W, *bias, *residual;   // [N,K], [N], [rows,N]
    float *out;                         // [rows,N]
    int rows, N, K, relu;
};

// out = relu(LN(x) W^T + bias) + residual for up to 16 MT rows.  A workgroup takes 16 columns; its waves share K, 64
// at a time, and add up in LDS.  fp32 matrix instructions: lane (g, c) holds 4 consecutive k of row c as one 16-byte load
// of either operand, and register r of the two is the r-th instruction's k (the sum over k does not mind its order).
// Bound by latency: one round trip to the weights, then the sum over waves (4.4 us a call of which 2.4 are an empty kernel's;
// with the bias, residual and LayerNorm weights fetched where they are used 5.7).
template <int MT, bool LN>
__global__ __launch_bounds__(1024) void k_rows(RowsArgs a) {
    extern __shared__ float lds[];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, waves = blockDim.x / 64;
    const int c = lane % 16, g = lane / 16, n = min((int)blockIdx.x * 16 + c, a.N - 1);
    v4f acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};
    // what the end needs, asked for at the start: a trip to memory is a third of such a kernel
    const int col = blockIdx.x * 16 + c;
    float bias = 0.f, res[4] = {0.f, 0.f, 0.f, 0.f};
    if (wave < MT && col < a.N) {
        if (a.bias) bias = a.bias[col];
        if (a.residual)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int row = 16 * wave + 4 * g + r;
                if (row < a.rows) res[r] = a.residual[(int64_t)row * a.N + col];
            }
    }
    // LN: exactly once per wave, also for a wave beyond K (it meets the barriers and adds zeros)
    for (int k0 = 64 * wave; LN || k0 < a.K; k0 += 64 * waves) {
        v4f w[4], x[MT][4];
        const bool valid = k0 < a.K;
        const int k = (valid ? k0 : 0) + 4 * g;
#pragma unroll
        for (int s = 0; s < 4; s++) w[s] = ld4(a.W + (int64_t)n * a.K + k + 16 * s);
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int s = 0; s < 4; s++) x[t][s] = ld4(a.x + (int64_t)min(16 * t + c, a.rows - 1) * a.K + k + 16 * s);
        if constexpr (LN) {
            v4f gam[4], bet[4];
#pragma unroll
            for (int s = 0; s < 4; s++) gam[s] = ld4(a.gamma + k + 16 * s), bet[s] = ld4(a.beta + k + 16 * s);
            float mean[MT];
            // a row's values sit in the four lanes (g, c), g = 0..3, of every wave
            const auto row_sums = [&](float (&v)[MT]) {
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    v[t] += __shfl_xor(v[t], 16, 64);
                    v[t] += __shfl_xor(v[t], 32, 64);
                    if (g == 0) lds[wave * 16 * MT + 16 * t + c] = v[t];
                }
                __syncthreads();
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    v[t] = 0.f;
                    for (int i = 0; i < waves; i++) v[t] += lds[i * 16 * MT + 16 * t + c];
                    v[t] /= a.K;
                }
                __syncthreads();
            };
#pragma unroll
            for (int t = 0; t < MT; t++) {
                mean[t] = 0.f;
#pragma unroll
                for (int s = 0; s < 4; s++) mean[t] += (x[t][s][0] + x[t][s][1]) + (x[t][s][2] + x[t][s][3]);
                if (!valid) mean[t] = 0.f;
            }
            row_sums(mean);
            float var[MT];
#pragma unroll
            for (int t = 0; t < MT; t++) {
                var[t] = 0.f;
#pragma unroll
                for (int s = 0; s < 4; s++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        x[t][s][r] -= mean[t];
                        var[t] += x[t][s][r] * x[t][s][r];
                    }
                if (!valid) var[t] = 0.f;
            }
            row_sums(var);
#pragma unroll
            for (int s = 0; s < 4; s++) {
#pragma unroll
                for (int t = 0; t < MT; t++) {
                    const float rstd = 1.f / sqrtf(var[t] + a.eps);
#pragma unroll
                    for (int r = 0; r < 4; r++) x[t][s][r] = valid ? x[t][s][r] * rstd * gam[s][r] + bet[s][r] : 0.f;
                    if (a.y && valid && blockIdx.x == 0 && 16 * t + c < a.rows)
                        *reinterpret_cast<v4f *>(a.y + (int64_t)(16 * t + c) * a.K + k + 16 * s) = x[t][s];
                }
            }
        }
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int t = 0; t < MT; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[t][s][r], w[s][r], acc[t], 0, 0, 0);
        if (LN) break;
    }
    // acc[t][r] = row 16 t + 4 g + r, column c of the workgroup's 16
    v4f *const red = reinterpret_cast<v4f *>(lds);
#pragma unroll
    for (int t = 0; t < MT; t++) red[(wave * MT + t) * 64 + lane] = acc[t];
    __syncthreads();
    // wave t adds up rows 16 t .. (four waves at least when there are more than 32 rows to add up, see rows_matmul)
    if (wave >= MT || col >= a.N) return;
    v4f v = red[wave * 64 + lane];
    for (int i = 1; i < waves; i++) v += red[(i * MT + wave) * 64 + lane];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int row = 16 * wave + 4 * g + r;
        if (row >= a.rows) continue;
        float o = v[r] + bias;
        if (a.relu) o = relu(o);
        a.out[(int64_t)row * a.N + col] = o + res[r];
    }
}

// The layer's pre-step and the delta rule's single step (fwp_layer.hip, fwp_step.hip) from one row of the projection:
// one wave per (sequence, head), the state read from `from` (NULL: zero) and written to `to`.
template <int D>
__global__ __launch_bounds__(64) void k_layer_step(const float *__restrict__ qkvb, const float *__restrict__ from,
                                                   float *__restrict__ to, float *__restrict__ out, float q_scale) {
    constexpr int CG = D / 4, RG = 64 / CG, RI = D / RG;
    const int lane = threadIdx.x, cg = lane % CG, rg = lane / CG;
    const int64_t seq = blockIdx.x;
    const float *src = qkvb + seq * (3 * D + 1);
    const auto over_rows = [](float x) {
#pragma unroll
        for (int m = CG; m < 64; m *= 2) x += __shfl_xor(x, m, 64);
        return x;
    };
    const auto feature = [](float x) { return x > 0.f ? x + 1.f : __expf(x); };      // elu(x) + 1
    v4f w[RI];
    float q[RI], k[RI], sq = 0.f, sk = 0.f;
#pragma unroll
    for (int i = 0; i < RI; i++) {
        const int row = rg + RG * i;
        w[i] = from ? ld4(from + (seq * D + row) * D + 4 * cg) : v4f{0.f, 0.f, 0.f, 0.f};
        q[i] = feature(src[row]);
        k[i] = feature(src[D + row]);
        sq += q[i];
        sk += k[i];
    }
    const float *vp = src + 2 * D + 4 * cg;
    const v4f v = {vp[0], vp[1], vp[2], vp[3]};
    const float b = 1.f / (1.f + __expf(-src[3 * D]));
    sq = over_rows(sq);
    sk = over_rows(sk);
    v4f old = {0.f, 0.f, 0.f, 0.f}, read = old;
    float kq = 0.f;
#pragma unroll
    for (int i = 0; i < RI; i++) {
        q[i] = q[i] / sq * q_scale;
        k[i] = k[i] / sk;
        old += k[i] * w[i];
        read += q[i] * w[i];
        kq += k[i] * q[i];
    }
#pragma unroll
    for (int e = 0; e < 4; e++) old[e] = over_rows(old[e]), read[e] = over_rows(read[e]);
    kq = over_rows(kq);
    const v4f u = b * (v - old);
#pragma unroll
    for (int i = 0; i < RI; i++) *reinterpret_cast<v4f *>(to + (seq * D + rg + RG * i) * D + 4 * cg) = w[i] + k[i] * u;
    if (rg == 0) *reinterpret_cast<v4f *>(out + seq * D + 4 * cg) = read + kq * u;
}

// out[t,b,:] = table[ids[t,b]] * scale + [sin | cos](position(t) inv_freq), positions counting down to zero at the
// newest token.  An id outside the table gives NaN.
__global__ __launch_bounds__(256) void k_embed(const float *__restrict__ table, const int64_t *__restrict__ ids,
                                               const float *__restrict__ inv_freq, float *__restrict__ out, int T, int B, int d,
                                               int64_t n_token, float scale, float clamp) {
    const int64_t at = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (at >= (int64_t)T * B * d) return;
    const int64_t row = at / d;
    const int j = (int)(at % d), half = d / 2;
    const int64_t id = ids[row];
    float pos = (float)(T - 1 - row / B);
    if (clamp > 0.f) pos = fminf(pos, clamp);
    const float phase = pos * inv_freq[j < half ? j : j - half];
    const float e = id >= 0 && id < n_token ? table[id * d + j] : NAN;
    out[at] = __fadd_rn(__fmul_rn(e, scale), j < half ? sinf(phase) : cosf(phase));      // rounded as two operations
}

}  // namespace

bool rows_supported(int rows, int K, bool norm) { return rows >= 1 && rows <= 64 && K >= 64 && K % 64 == 0 && (!norm || K <= 1024); }

int rows_matmul(const float *x, const float *gamma, const float *beta, float eps, float *y, const float *W, const float *bias,
                const float *residual, int relu, float *out, int rows, int N, int K, hipStream_t s) {
    const RowsArgs a = {x, gamma, beta, eps, y, W, bias, residual, out, rows, N, K, relu};
    const int mt = rows <= 16 ? 1 : rows <= 32 ? 2 : 4;
    int waves = K / 64 < 16 ? K / 64 : 16;
    if (waves < mt) waves = mt;         // a wave per 16 rows at the end (those beyond K / 64 add zeros)
    const dim3 grid((N + 15) / 16), block(64 * waves);
    const size_t bytes = (size_t)waves * mt * 1024;
#define FWP_ROWS(MT)                                                                              \
    do {                                                                                          \
        if (gamma) hipLaunchKernelGGL((k_rows<MT, true>), grid, block, bytes, s, a);              \
        else hipLaunchKernelGGL((k_rows<MT, false>), grid, block, bytes, s, a);                   \
    } while (0)
    if (mt == 1) FWP_ROWS(1);
    else if (mt == 2) FWP_ROWS(2);
    else FWP_ROWS(4);
#undef FWP_ROWS
    return (int)hipGetLastError();
}

int layer_step(const float *qkvb, const float *from, float *to, float *out, int B, int H, int D, float q_scale, hipStream_t s) {
    const dim3 grid(B * H);
    if (D == 16) hipLaunchKernelGGL(k_layer_step<16>, grid, dim3(64), 0, s, qkvb, from, to, out, q_scale);
    else if (D == 32) hipLaunchKernelGGL(k_layer_step<32>, grid, dim3(64), 0, s, qkvb, from, to, out, q_scale);
    else hipLaunchKernelGGL(k_layer_step<64>, grid, dim3(64), 0, s, qkvb, from, to, out, q_scale);
    return (int)hipGetLastError();
}

int embed(const float *table, const int64_t *ids, const float *inv_freq, float *out, int T, int B, int d, int64_t n_token,
          float scale, float clamp, hipStream_t s) {
    const int64_t total = (int64_t)T * B * d;
    hipLaunchKernelGGL(k_embed, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, table, ids, inv_freq, out, T, B, d, n_token,
                       scale, clamp);
    return (int)hipGetLastError();
}

}  // namespace fwp
