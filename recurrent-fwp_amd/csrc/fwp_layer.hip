// Fused pre-step of the Delta-Net layer (reference: language_modeling/src/utils/
// cuda_fast_weight_layer.py:108-125): from the layer's one projection qkvb[T,B,H,3D+1] straight to
// the operator's inputs in [B,H,T,.] order,
//     q, k = (elu(x) + 1) / sum_D(elu(x) + 1)      v = copy      beta = sigmoid
// (q times a constant on request: the operator's output is linear in q, so the 1/sqrt(D) the layer
// applies to that output can be applied here, to D values per token instead of a pass of its own)
// and its adjoint: one pass over the data each way instead of the dozen elementwise, reduction
// and copy kernels the same lines cost in stock PyTorch.
//
// Bound by HBM: two passes over T B H (3D+1) floats forward, three backward.  A lane takes four columns of a row
// (16-byte loads at the 4-byte alignment that rows of 3D+1 floats have), D/4 lanes a row, so that a row's sum is two to
// four DPP moves, and a workgroup takes up to eight heads of consecutive steps: it reads whole tokens and writes
// 512 bytes or more of a head's sequence at once, and finds its place by shifts.  With D lanes to a row and a
// workgroup's rows in the order of qkvb, three 64-bit divisions a row and ten shuffles bounded both passes.  32 x 1024 tokens of 8
// heads of 32: forward 45.2 -> 31.6 us (6.4 TB/s), backward 71.7 -> 53.8 us (5.7 TB/s); 96 x 256 tokens of 8 heads of
// 16: 16.4 -> 13.0 and 23.2 -> 20.8 us.  Up to about 2000 tokens both are as long as a launch.
#include "fwp_common.hpp"
#include "fwp_wave.hpp"

namespace fwp {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

// Four values at any address of a float: the rows of qkvb are 3D+1 long.
struct __attribute__((packed, aligned(4))) Any4 { v4f x; };
__device__ __forceinline__ v4f load(const float *p) { return reinterpret_cast<const Any4 *>(p)->x; }
__device__ __forceinline__ void store(float *p, v4f x) { reinterpret_cast<Any4 *>(p)->x = x; }

// The sum over the D/4 lanes of a row, in all of them: columns D/2 apart first, then D/4 ... 1, the order in which one lane to a column would
// exchange them.  (Another order rounds as well, but where the results lie close to zero a rectifier behind may turn.)
template <int D>
__device__ __forceinline__ float row_sum(v4f y) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
        y[i] += dpp<kQuadXor1>(y[i]);
        y[i] += dpp<kQuadXor2>(y[i]);
        if constexpr (D >= 32) y[i] += dpp<0x141>(y[i]);      // row_half_mirror: the quads' lanes are alike by now
        if constexpr (D >= 64) y[i] += dpp<0x140>(y[i]);      // row_mirror
    }
    return (y.x + y.z) + (y.y + y.w);
}

// The first of lane l's four columns: the bits of l the other way round, as row_sum wants them
template <int D>
__device__ __forceinline__ int column_of(int l) {
    return D == 16 ? (l & 1) * 8 + (l >> 1) * 4 : D == 32 ? (l & 1) * 16 + (l & 2) * 4 + (l >> 2) * 4 : (l & 1) * 32 + (l & 2) * 8 + (l & 4) * 2 + (l >> 3) * 4;
}

__device__ __forceinline__ float feature(float x) { return x > 0.f ? x + 1.f : __expf(x); }   // elu(x) + 1
__device__ __forceinline__ v4f feature(v4f x) { return v4f{feature(x.x), feature(x.y), feature(x.z), feature(x.w)}; }

// The sizes, and a workgroup's rows: 1 << h heads of 1 << t steps of 1 << b sequences
struct Tile { int T, B, H, h, t, b; };

constexpr int kThreads = 256;

// The row that this lane works on: its number in (t, b, h) order and in (b, h, t) order, and its first column.
struct Row {
    int64_t in, out;
    int col;
    bool ok;
    template <int D> static __device__ __forceinline__ Row of(const Tile &a) {
        const int lanes = D / 4, i = threadIdx.x / lanes;
        const unsigned nh = ((unsigned)a.H + (1u << a.h) - 1) >> a.h, nt = ((unsigned)a.T + (1u << a.t) - 1) >> a.t;
        const unsigned w = blockIdx.x / nh;
        const int h = (int)((blockIdx.x % nh) << a.h) + (i & ((1 << a.h) - 1));
        const int t = (int)((w % nt) << a.t) + (i >> a.h & ((1 << a.t) - 1));
        const int b = (int)((w / nt) << a.b) + (i >> (a.h + a.t));
        return {((int64_t)t * a.B + b) * a.H + h, ((int64_t)b * a.H + h) * a.T + t, column_of<D>(threadIdx.x % lanes),
                t < a.T && b < a.B && h < a.H};
    }
};

// zeros: 16-byte groups of the state that the operator behind starts from; a fill of its own was 2.3 us a layer (2381 tokens) to 4.7 (32768).
template <int D>
__global__ __launch_bounds__(kThreads) void k_prep_fwd(const float *__restrict__ qkvb, float *__restrict__ q,
                                                       float *__restrict__ k, float *__restrict__ v,
                                                       float *__restrict__ beta, float *__restrict__ zero, int64_t zeros,
                                                       Tile a, float q_scale) {
    for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < zeros; i += (int64_t)gridDim.x * kThreads) store(zero + 4 * i, v4f{0.f, 0.f, 0.f, 0.f});
    const Row r = Row::of<D>(a);
    if (!r.ok) return;              // all lanes of a row together
    const float *src = qkvb + r.in * (3 * D + 1);
    const v4f xq = load(src + r.col), xk = load(src + D + r.col), xv = load(src + 2 * D + r.col);
    const float xb = src[3 * D];
    const v4f fq = feature(xq), fk = feature(xk);
    const float sq = row_sum<D>(fq), sk = row_sum<D>(fk);
    const int64_t o = r.out * D + r.col;
    store(q + o, fq / sq * q_scale);
    store(k + o, fk / sk);
    store(v + o, xv);
    if (r.col == 0) beta[r.out] = 1.f / (1.f + __expf(-xb));
}

template <int D>
__global__ __launch_bounds__(kThreads) void k_prep_bwd(const float *__restrict__ qkvb,
                                                       const float *__restrict__ gq,
                                                       const float *__restrict__ gk,
                                                       const float *__restrict__ gv,
                                                       const float *__restrict__ gbeta,
                                                       float *__restrict__ gqkvb, Tile a, float q_scale) {
    const Row r = Row::of<D>(a);
    if (!r.ok) return;
    const float *src = qkvb + r.in * (3 * D + 1);
    float *dst = gqkvb + r.in * (3 * D + 1);
    const int64_t o = r.out * D + r.col;
    // y = f / s with f = elu(x) + 1, s = sum f:  dx = (dy - sum(dy y)) / s * f'(x),  f' = 1 (x > 0) or f
    const v4f xq = load(src + r.col), xk = load(src + D + r.col);
    const v4f dq = load(gq + o) * q_scale, dk = load(gk + o), dv = load(gv + o);
    const float xb = src[3 * D], db = gbeta[r.out];
    const v4f fq = feature(xq), fk = feature(xk);
    const float sq = row_sum<D>(fq), sk = row_sum<D>(fk);
    const float cq = row_sum<D>(dq * fq) / sq, ck = row_sum<D>(dk * fk) / sk;      // sum(dy y)
    v4f yq = (dq - cq) / sq, yk = (dk - ck) / sk;
#pragma unroll
    for (int i = 0; i < 4; i++) yq[i] *= xq[i] > 0.f ? 1.f : fq[i], yk[i] *= xk[i] > 0.f ? 1.f : fk[i];
    store(dst + r.col, yq);
    store(dst + D + r.col, yk);
    store(dst + 2 * D + r.col, dv);
    if (r.col == 0) {
        const float s = 1.f / (1.f + __expf(-xb));
        dst[3 * D] = db * s * (1.f - s);
    }
}

int log2_up(int n, int most) {
    int l = 0;
    while (l < most && (1 << l) < n) l++;
    return l;
}

// Eight heads make the reads whole lines but for a token's ends and leave room for the steps that the writes need; what
// few heads or few steps leave of the workgroup goes to other sequences.
Tile tile_of(int T, int B, int H, int D) {
    const int rows = D == 16 ? 6 : D == 32 ? 5 : 4;     // log2 of a workgroup's rows
    const int h = log2_up(H, 3), t = log2_up(T, rows - h);
    return {T, B, H, h, t, rows - h - t};
}

dim3 grid_of(const Tile &a) {
    const auto n = [](int size, int l) { return ((int64_t)size + (1 << l) - 1) >> l; };
    return dim3((unsigned)(n(a.H, a.h) * n(a.T, a.t) * n(a.B, a.b)));
}

}  // namespace

bool prep_supported(int D) { return D == 16 || D == 32 || D == 64; }

int deltanet_prep_fwd(const float *qkvb, float *q, float *k, float *v, float *beta, float *state, int T, int B, int H,
                      int D, float q_scale, hipStream_t s) {
    const Tile a = tile_of(T, B, H, D);
    const int64_t zeros = state ? (int64_t)B * H * D * D / 4 : 0;
    const dim3 grid = grid_of(a), block(kThreads);
    if (D == 16) hipLaunchKernelGGL(k_prep_fwd<16>, grid, block, 0, s, qkvb, q, k, v, beta, state, zeros, a, q_scale);
    else if (D == 32) hipLaunchKernelGGL(k_prep_fwd<32>, grid, block, 0, s, qkvb, q, k, v, beta, state, zeros, a, q_scale);
    else hipLaunchKernelGGL(k_prep_fwd<64>, grid, block, 0, s, qkvb, q, k, v, beta, state, zeros, a, q_scale);
    return (int)hipGetLastError();
}

int deltanet_prep_bwd(const float *qkvb, const float *gq, const float *gk, const float *gv,
                      const float *gbeta, float *gqkvb, int T, int B, int H, int D, float q_scale, hipStream_t s) {
    const Tile a = tile_of(T, B, H, D);
    const dim3 grid = grid_of(a), block(kThreads);
    if (D == 16) hipLaunchKernelGGL(k_prep_bwd<16>, grid, block, 0, s, qkvb, gq, gk, gv, gbeta, gqkvb, a, q_scale);
    else if (D == 32) hipLaunchKernelGGL(k_prep_bwd<32>, grid, block, 0, s, qkvb, gq, gk, gv, gbeta, gqkvb, a, q_scale);
    else hipLaunchKernelGGL(k_prep_bwd<64>, grid, block, 0, s, qkvb, gq, gk, gv, gbeta, gqkvb, a, q_scale);
    return (int)hipGetLastError();
}

}  // namespace fwp
