/*
 * A stand-in for libfwp_hip.so on a machine without a GPU: every entry point of include/fwp_hip.h, with
 * HOST pointers.  Nothing is launched; each call READS every element of its inputs through their views
 * and WRITES every element of its outputs and saved buffers (simple sums, so that results depend on the
 * inputs), which is what makes it useful under AddressSanitizer: a buffer of the wrong size, a view of
 * freed memory or a stride mistake in the host binding above it (csrc/fwp_torch*.cpp built with
 * -DFWP_HOST_STUB) shows up as a report instead of passing unseen.  The language model's products, LayerNorm, loss
 * and embedding are computed, one element after the other, so that the blocks made of them can be compared
 * with PyTorch's operators.  Test infrastructure only.
 */
#include <math.h>
#include <stddef.h>
#include <stdlib.h>
#include <string.h>

#include "fwp_hip.h"

static int g_calls;
int fwp_stub_calls(void) { return g_calls; }

static double sum_view(fwp_view v, int N, int H, int L, int D) {
    double s = 0;
    for (int n = 0; n < N; n++)
        for (int h = 0; h < H; h++)
            for (int l = 0; l < L; l++) {
                const float *r = v.ptr + n * v.sN + h * v.sH + l * v.sL;
                for (int d = 0; d < D; d++) s += r[d];
            }
    return s;
}
static double sum_flat(const float *p, long long n) {
    double s = 0;
    for (long long i = 0; i < n; i++) s += p[i];
    return s;
}
static void fill(float *p, long long n, double x) {
    for (long long i = 0; i < n; i++) p[i] = (float)(x + 1e-3 * (double)(i % 97));
}
static void bump(float *p, long long n) {
    for (long long i = 0; i < n; i++) p[i] += 1.0f;
}

const char *fwp_strerror(int code) { return code ? "stub error" : "ok"; }
int fwp_query(int what) {
    switch (what) {
        case FWP_Q_VERSION: return 2;
        case FWP_Q_CHUNK_QUANTUM: return 32;
        case FWP_Q_DEFAULT_CHUNK: return 64;
        case FWP_Q_MAX_STATE_FLOATS: return 16384;
        case FWP_Q_STATIC_SCRATCH_FLOATS: return 2 << 20;
        default: return 64;
    }
}
int fwp_config(int key, int value) { (void)key; (void)value; return 0; }
int fwp_check_device(void) { return 0; }
int fwp_delta_kind(int backward, fwp_view q, fwp_view k, fwp_view x, fwp_view beta, int N, int H, int L,
                   int E, int M) {
    (void)backward; (void)q; (void)k; (void)x; (void)beta; (void)N; (void)H; (void)L; (void)E; (void)M;
    return FWP_KIND_LDS;
}
int fwp_delta_fwd_kind(fwp_view q, fwp_view k, fwp_view v, fwp_view beta, fwp_out_view out, int saves, int N,
                       int H, int L, int E, int M) {
    (void)q; (void)k; (void)v; (void)beta; (void)out; (void)saves; (void)N; (void)H; (void)L; (void)E; (void)M;
    return FWP_KIND_LDS;
}
static long long nchunk(int L, int chunk) { return (L + chunk - 1) / chunk; }
long long fwp_delta_ckpt_floats(int N, int H, int L, int E, int M, int chunk) {
    if (N < 1 || H < 1 || L < 1 || E < 1 || M < 1 || chunk < 1) return -1;
    /* the states, a header and one 16 x 16 matrix per 16 steps, as the real library sizes it */
    return (long long)N * H * nchunk(L, chunk) * E * M + 64 + (long long)N * H * ((L + 15) / 16) * 256;
}

int fwp_delta_fwd_strided(fwp_view q, fwp_view k, fwp_view v, fwp_view beta, float *W, fwp_out_view out,
                          float *vdiff, float *ckpt, int N, int H, int L, int E, int M, int chunk, void *stream) {
    (void)stream;
    g_calls++;
    const double s = sum_view(q, N, H, L, E) + sum_view(k, N, H, L, E) + sum_view(v, N, H, L, M) +
                     sum_view(beta, N, H, L, 1) + sum_flat(W, (long long)N * H * E * M);
    for (int n = 0; n < N; n++)
        for (int h = 0; h < H; h++)
            for (int l = 0; l < L; l++) fill(out.ptr + n * out.sN + h * out.sH + l * out.sL, M, s);
    bump(W, (long long)N * H * E * M);
    if (vdiff) fill(vdiff, (long long)N * H * L * M, s);
    if (ckpt) fill(ckpt, fwp_delta_ckpt_floats(N, H, L, E, M, chunk), s);
    return 0;
}
/* a sequence of 256 steps or more is "cut": the call's scratch is overwritten to its end */
long long fwp_delta_segment_floats(int N, int H, int L, int E, int M, int chunk) {
    (void)chunk;
    return L < 256 ? 0 : (long long)N * H * (L / 64) * (E * M + E * E);
}
long long fwp_delta_bwd_segment_floats(int N, int H, int L, int E, int M, int chunk) {
    return L < 320 ? 0 : fwp_delta_segment_floats(N, H, L, E, M, chunk) - 1;
}
int fwp_delta_fwd_segments(fwp_view q, fwp_view k, fwp_view v, fwp_view beta, float *W, fwp_out_view out, float *vdiff,
                           float *ckpt, float *work, int N, int H, int L, int E, int M, int chunk, void *stream) {
    if (work) fill(work, fwp_delta_segment_floats(N, H, L, E, M, chunk), 1);
    return fwp_delta_fwd_strided(q, k, v, beta, W, out, vdiff, ckpt, N, H, L, E, M, chunk, stream);
}
int fwp_delta_fwd(fwp_view q, fwp_view k, fwp_view v, fwp_view beta, float *W, float *out, float *vdiff,
                  float *ckpt, int N, int H, int L, int E, int M, int chunk, void *stream) {
    fwp_out_view ov = {out, (int64_t)H * L * M, (int64_t)L * M, M};
    return fwp_delta_fwd_strided(q, k, v, beta, W, ov, vdiff, ckpt, N, H, L, E, M, chunk, stream);
}
int fwp_delta_bwd(fwp_view q, fwp_view k, fwp_view beta, const float *vdiff, fwp_view grad_out,
                  const float *ckpt, float *gq, float *gk, float *gv, float *gbeta, int N, int H, int L, int E,
                  int M, int chunk, void *stream) {
    (void)stream;
    g_calls++;
    const long long T = (long long)N * H * L;
    const double s = sum_view(q, N, H, L, E) + sum_view(k, N, H, L, E) + sum_view(beta, N, H, L, 1) +
                     sum_view(grad_out, N, H, L, M) + sum_flat(vdiff, T * M) +
                     sum_flat(ckpt, fwp_delta_ckpt_floats(N, H, L, E, M, chunk));
    fill(gq, T * E, s);
    fill(gk, T * E, s + 1);
    fill(gv, T * M, s + 2);
    fill(gbeta, T, s + 3);
    return 0;
}
int fwp_delta_bwd_segments(fwp_view q, fwp_view k, fwp_view beta, const float *vdiff, fwp_view grad_out,
                           const float *ckpt, float *gq, float *gk, float *gv, float *gbeta, float *work, int N, int H, int L,
                           int E, int M, int chunk, void *stream) {
    if (work) fill(work, fwp_delta_bwd_segment_floats(N, H, L, E, M, chunk), 1);
    return fwp_delta_bwd(q, k, beta, vdiff, grad_out, ckpt, gq, gk, gv, gbeta, N, H, L, E, M, chunk, stream);
}

int fwp_sum_fwd(fwp_view q, fwp_view k, fwp_view v, float *W, float *out, float *ckpt, int N, int H, int L,
                int E, int M, int chunk, void *stream) {
    (void)stream;
    g_calls++;
    const double s = sum_view(q, N, H, L, E) + sum_view(k, N, H, L, E) + sum_view(v, N, H, L, M) +
                     sum_flat(W, (long long)N * H * E * M);
    fill(out, (long long)N * H * L * M, s);
    bump(W, (long long)N * H * E * M);
    if (ckpt) fill(ckpt, (long long)N * H * nchunk(L, chunk) * E * M, s);
    return 0;
}
int fwp_sum_bwd(fwp_view q, fwp_view k, fwp_view v, fwp_view grad_out, const float *ckpt, const float *W_init,
                float *gq, float *gk, float *gv, int N, int H, int L, int E, int M, int chunk, void *stream) {
    (void)stream;
    g_calls++;
    const long long T = (long long)N * H * L;
    double s = sum_view(q, N, H, L, E) + sum_view(k, N, H, L, E) + sum_view(v, N, H, L, M) +
               sum_view(grad_out, N, H, L, M) + sum_flat(ckpt, (long long)N * H * nchunk(L, chunk) * E * M);
    if (W_init) s += sum_flat(W_init, (long long)N * H * E * M);
    fill(gq, T * E, s);
    fill(gk, T * E, s + 1);
    fill(gv, T * M, s + 2);
    return 0;
}

int fwp_rnn_fwd(fwp_view z, fwp_view k, fwp_view v, fwp_view beta, float *W, float *h, float *out, float *vdiff,
                float *ckpt, int N, int H, int L, int D, int chunk, void *stream) {
    (void)stream;
    g_calls++;
    const long long T = (long long)N * H * L;
    const double s = sum_view(z, N, H, L, D) + sum_view(k, N, H, L, D) + sum_view(v, N, H, L, D) +
                     sum_view(beta, N, H, L, 1) + sum_flat(W, (long long)N * H * D * D) +
                     sum_flat(h, (long long)N * H * D);
    fill(out, T * D, s);
    bump(W, (long long)N * H * D * D);
    bump(h, (long long)N * H * D);
    if (vdiff) fill(vdiff, T * D, s);
    if (ckpt) fill(ckpt, (long long)N * H * nchunk(L, chunk) * D * D, s);
    return 0;
}
int fwp_rnn_bwd(fwp_view k, fwp_view beta, const float *vdiff, const float *out, const float *h_init,
                fwp_view grad_out, const float *ckpt, float *gz, float *gk, float *gv, float *gbeta, int N,
                int H, int L, int D, int chunk, void *stream) {
    (void)stream;
    g_calls++;
    const long long T = (long long)N * H * L;
    const double s = sum_view(k, N, H, L, D) + sum_view(beta, N, H, L, 1) + sum_view(grad_out, N, H, L, D) +
                     sum_flat(vdiff, T * D) + sum_flat(out, T * D) + sum_flat(h_init, (long long)N * H * D) +
                     sum_flat(ckpt, (long long)N * H * nchunk(L, chunk) * D * D);
    fill(gz, T * D, s);
    fill(gk, T * D, s + 1);
    fill(gv, T * D, s + 2);
    fill(gbeta, T, s + 3);
    return 0;
}

int fwp_lstm_fwd(const fwp_view *z, const fwp_view *k, const fwp_view *v, const fwp_view *beta, float *const *W,
                 float *h, float *c, float *out, float *cell, float *gates, float *vdiff, float *ckpt, int N,
                 int H, int L, int D, int chunk, void *stream) {
    (void)stream;
    g_calls++;
    const long long T = (long long)N * H * L;
    double s = sum_flat(h, (long long)N * H * D) + sum_flat(c, (long long)N * H * D);
    for (int a = 0; a < 3; a++) {
        s += sum_view(z[a], N, H, L, D) + sum_view(k[a], N, H, L, D) + sum_view(v[a], N, H, L, D) +
             sum_view(beta[a], N, H, L, 1) + sum_flat(W[a], (long long)N * H * D * D);
        bump(W[a], (long long)N * H * D * D);
    }
    fill(out, T * D, s);
    fill(cell, T * D, s + 1);
    bump(h, (long long)N * H * D);
    bump(c, (long long)N * H * D);
    if (gates) fill(gates, 3 * T * D, s);
    if (vdiff) fill(vdiff, 3 * T * D, s);
    if (ckpt) fill(ckpt, 3LL * N * H * nchunk(L, chunk) * D * D, s);
    return 0;
}
int fwp_lstm_bwd(const fwp_view *k, const fwp_view *beta, const float *vdiff, const float *gates,
                 const float *out, const float *cell, const float *h_init, const float *c_init,
                 fwp_view grad_out, const float *ckpt, float *gz, float *gk, float *gv, float *gbeta, int N,
                 int H, int L, int D, int chunk, void *stream) {
    (void)stream;
    g_calls++;
    const long long T = (long long)N * H * L;
    double s = sum_view(grad_out, N, H, L, D) + sum_flat(vdiff, 3 * T * D) + sum_flat(gates, 3 * T * D) +
               sum_flat(out, T * D) + sum_flat(cell, T * D) + sum_flat(h_init, (long long)N * H * D) +
               sum_flat(c_init, (long long)N * H * D) + sum_flat(ckpt, 3LL * N * H * nchunk(L, chunk) * D * D);
    for (int a = 0; a < 3; a++) s += sum_view(k[a], N, H, L, D) + sum_view(beta[a], N, H, L, 1);
    fill(gz, 3 * T * D, s);
    fill(gk, 3 * T * D, s + 1);
    fill(gv, 3 * T * D, s + 2);
    fill(gbeta, 3 * T, s + 3);
    return 0;
}

int fwp_deltanet_prep_fwd(const float *qkvb, float *q, float *k, float *v, float *beta, int T, int B, int H,
                          int D, float q_scale, void *stream) {
    (void)stream;
    g_calls++;
    const long long R = (long long)T * B * H;
    const double s = sum_flat(qkvb, R * (3 * D + 1)) + q_scale;
    fill(q, R * D, s);
    fill(k, R * D, s);
    fill(v, R * D, s);
    fill(beta, R, s);
    return 0;
}
int fwp_deltanet_prep_start(const float *qkvb, float *q, float *k, float *v, float *beta, float *state, int T, int B,
                            int H, int D, float q_scale, void *stream) {
    fill(state, (long long)B * H * D * D, 0);
    return fwp_deltanet_prep_fwd(qkvb, q, k, v, beta, T, B, H, D, q_scale, stream);
}
int fwp_deltanet_prep_bwd(const float *qkvb, const float *gq, const float *gk, const float *gv,
                          const float *gbeta, float *gqkvb, int T, int B, int H, int D, float q_scale,
                          void *stream) {
    (void)stream;
    g_calls++;
    const long long R = (long long)T * B * H;
    const double s = sum_flat(qkvb, R * (3 * D + 1)) + sum_flat(gq, R * D) + sum_flat(gk, R * D) +
                     sum_flat(gv, R * D) + sum_flat(gbeta, R) + q_scale;
    fill(gqkvb, R * (3 * D + 1), s);
    return 0;
}

int fwp_rec_fwd(fwp_view qx, fwp_view kx, fwp_view vx, fwp_view bx, const float *Rq, const float *Rk,
                const float *Rv, const float *rb, float *W, float *h, float *out, float *q_act, float *k_act,
                float *beta_act, float *vdiff, float *ckpt, int N, int H, int L, int D, int chunk, void *stream) {
    (void)stream;
    g_calls++;
    const long long T = (long long)N * H * L;
    const double s = sum_view(qx, N, H, L, D) + sum_view(kx, N, H, L, D) + sum_view(vx, N, H, L, D) +
                     sum_view(bx, N, H, L, 1) + sum_flat(Rq, (long long)H * D * D) +
                     sum_flat(Rk, (long long)H * D * D) + sum_flat(Rv, (long long)H * D * D) +
                     sum_flat(rb, (long long)H * D) + sum_flat(W, (long long)N * H * D * D) +
                     sum_flat(h, (long long)N * H * D);
    fill(out, T * D, s);
    bump(W, (long long)N * H * D * D);
    bump(h, (long long)N * H * D);
    if (q_act) fill(q_act, T * D, s);
    if (k_act) fill(k_act, T * D, s);
    if (beta_act) fill(beta_act, T, s);
    if (vdiff) fill(vdiff, T * D, s);
    if (ckpt) fill(ckpt, (long long)N * H * nchunk(L, chunk) * D * D, s);
    return 0;
}
static int rec_bwd(const float *q_act, const float *k_act, const float *beta_act, const float *vdiff,
                   const float *out, const float *h_init, fwp_view grad_out, const float *Rq, const float *Rk,
                   const float *Rv, const float *rb, const float *ckpt, float *gqx, float *gkx, float *gvx,
                   float *gbx, float *gRq, float *gRk, float *gRv, float *grb, float *workspace, int N, int H,
                   int L, int D, int chunk) {
    g_calls++;
    const long long T = (long long)N * H * L;
    const double s = sum_flat(q_act, T * D) + sum_flat(k_act, T * D) + sum_flat(beta_act, T) +
                     sum_flat(vdiff, T * D) + sum_flat(out, T * D) + sum_flat(h_init, (long long)N * H * D) +
                     sum_view(grad_out, N, H, L, D) + sum_flat(Rq, (long long)H * D * D) +
                     sum_flat(Rk, (long long)H * D * D) + sum_flat(Rv, (long long)H * D * D) +
                     sum_flat(rb, (long long)H * D) + sum_flat(ckpt, (long long)N * H * nchunk(L, chunk) * D * D);
    if (workspace) fill(workspace, (long long)N * H * (3 * D * D + D), s);
    fill(gqx, T * D, s);
    fill(gkx, T * D, s + 1);
    fill(gvx, T * D, s + 2);
    fill(gbx, T, s + 3);
    fill(gRq, (long long)H * D * D, s + 4);
    fill(gRk, (long long)H * D * D, s + 5);
    fill(gRv, (long long)H * D * D, s + 6);
    fill(grb, (long long)H * D, s + 7);
    return 0;
}
int fwp_rec_bwd(const float *q_act, const float *k_act, const float *beta_act, const float *vdiff,
                const float *out, const float *h_init, fwp_view grad_out, const float *Rq, const float *Rk,
                const float *Rv, const float *rb, const float *ckpt, float *gqx, float *gkx, float *gvx,
                float *gbx, float *gRq, float *gRk, float *gRv, float *grb, float *workspace, int N, int H, int L,
                int D, int chunk, void *stream) {
    (void)stream;
    return rec_bwd(q_act, k_act, beta_act, vdiff, out, h_init, grad_out, Rq, Rk, Rv, rb, ckpt, gqx, gkx, gvx, gbx,
                   gRq, gRk, gRv, grb, workspace, N, H, L, D, chunk);
}
int fwp_rec_bwd_static(const float *q_act, const float *k_act, const float *beta_act, const float *vdiff,
                       const float *out, const float *h_init, fwp_view grad_out, const float *Rq, const float *Rk,
                       const float *Rv, const float *rb, const float *ckpt, float *gqx, float *gkx, float *gvx,
                       float *gbx, float *gRq, float *gRk, float *gRv, float *grb, int N, int H, int L, int D,
                       int chunk, void *stream) {
    (void)stream;
    return rec_bwd(q_act, k_act, beta_act, vdiff, out, h_init, grad_out, Rq, Rk, Rv, rb, ckpt, gqx, gkx, gvx, gbx,
                   gRq, gRk, gRv, grb, NULL, N, H, L, D, chunk);
}

/* ---- the language model's kernels, computed */

long long fwp_product_workspace(int M, int N, int K) { (void)M; (void)N; return K >= 64 ? 8 : 0; }
long long fwp_matmul_workspace(int M, int N, int K) { (void)M; (void)N; return K >= 64 ? 8 : 0; }
int fwp_matmul(int layout, const float *A, long long lda, const float *B, long long ldb, float *C, long long ldc, int M,
               int N, int K, const fwp_mm_epilogue *epi, float *workspace, void *stream) {
    (void)stream;
    g_calls++;
    const fwp_mm_epilogue none = {0}, e = epi ? *epi : none;
    if (workspace) fill(workspace, fwp_product_workspace(M, N, K), 0);
    for (int m = 0; m < M; m++)
        for (int n = 0; n < N; n++) {
            double s = 0;
            for (int k = 0; k < K; k++)
                s += (double)(layout == FWP_MM_TN ? A[k * lda + m] : A[m * lda + k]) *
                     (layout == FWP_MM_NT ? B[n * ldb + k] : B[k * ldb + n]);
            const long long at = m * ldc + n;
            if (e.bias) s += e.bias[n];
            if (e.relu) s = s < 0 ? 0 : s;
            if (e.residual) s += e.residual[at];
            if (e.gate && e.gate[at] <= 0) s = 0;
            C[at] = (float)s;
        }
    if (layout == FWP_MM_TN && e.colsum)
        for (int m = 0; m < M; m++) {
            double s = 0;
            for (int k = 0; k < K; k++) s += A[k * lda + m];
            e.colsum[m] = (float)s;
        }
    return 0;
}

/* x's row normalised; the two statistics where wanted */
static void norm_row(const float *x, const float *gamma, const float *beta, float *y, float *stats, int cols, double eps) {
    double mean = 0, var = 0;
    for (int c = 0; c < cols; c++) mean += x[c];
    mean /= cols;
    for (int c = 0; c < cols; c++) var += (x[c] - mean) * (x[c] - mean);
    const double rstd = 1 / sqrt(var / cols + eps);
    for (int c = 0; c < cols; c++) y[c] = (float)((x[c] - mean) * rstd * gamma[c] + beta[c]);
    if (stats) stats[0] = (float)mean, stats[1] = (float)rstd;
}
int fwp_layer_norm_fwd(const float *x, const float *gamma, const float *beta, float *y, float *stats, int rows, int cols,
                       float eps, void *stream) {
    (void)stream;
    g_calls++;
    for (long long r = 0; r < rows; r++)
        norm_row(x + r * cols, gamma, beta, y + r * cols, stats ? stats + 2 * r : NULL, cols, eps);
    return 0;
}
long long fwp_layer_norm_workspace(int rows, int cols) { (void)rows; return 2 * cols; }
int fwp_layer_norm_bwd(const float *gy, const float *x, const float *stats, const float *gamma, float *gx,
                       float *ggamma, float *gbeta, float *workspace, int rows, int cols, void *stream) {
    (void)stream;
    g_calls++;
    fill(workspace, fwp_layer_norm_workspace(rows, cols), 0);
    memset(ggamma, 0, sizeof(float) * cols);
    memset(gbeta, 0, sizeof(float) * cols);
    for (long long r = 0; r < rows; r++) {
        const float *d = gy + r * cols, *p = x + r * cols;
        const double mean = stats[2 * r], rstd = stats[2 * r + 1];
        double s = 0, t = 0;
        for (int c = 0; c < cols; c++) {
            const double h = (p[c] - mean) * rstd, g = (double)d[c] * gamma[c];
            ggamma[c] += (float)(d[c] * h);
            gbeta[c] += d[c];
            s += g / cols, t += g * h / cols;
        }
        for (int c = 0; c < cols; c++)
            gx[r * cols + c] = (float)(rstd * ((double)d[c] * gamma[c] - s - (p[c] - mean) * rstd * t));
    }
    return 0;
}

long long fwp_nll_workspace(int rows, int vocab) { (void)vocab; return rows; }
static int nll_fwd(const float *x, const float *W, const float *bias, const int64_t *target, float *logits, float *loss,
                   float *lse, float *stats, float *workspace, int rows, int vocab, int dim) {
    g_calls++;
    fill(workspace, fwp_nll_workspace(rows, vocab), 0);
    float *row = malloc(sizeof(float) * vocab);
    for (long long r = 0; r < rows; r++) {
        double s = 0, mx = -INFINITY;
        for (long long v = 0; v < vocab; v++) {
            double l = bias ? bias[v] : 0;
            for (int k = 0; k < dim; k++) l += (double)x[r * dim + k] * W[v * dim + k];
            row[v] = (float)l;
            mx = fmax(mx, row[v]);
        }
        for (long long v = 0; v < vocab; v++) s += exp(row[v] - mx);
        if (logits) memcpy(logits + r * vocab, row, sizeof(float) * vocab);
        if (lse) lse[r] = (float)(mx + log(s));
        if (stats) stats[2 * r] = (float)mx, stats[2 * r + 1] = (float)(1 / s);
        loss[r] = target[r] == -100 ? 0 : target[r] < 0 || target[r] >= vocab ? NAN : (float)(mx - row[target[r]] + log(s));
    }
    free(row);
    return 0;
}
int fwp_nll_fwd(const float *x, const float *W, const float *bias, const int64_t *target, float *logits, float *loss,
                float *lse, float *workspace, int rows, int vocab, int dim, void *stream) {
    (void)stream;
    return nll_fwd(x, W, bias, target, logits, loss, lse, NULL, workspace, rows, vocab, dim);
}
int fwp_nll_stats_fwd(const float *x, const float *W, const float *bias, const int64_t *target, float *logits, float *loss,
                      float *stats, float *workspace, int rows, int vocab, int dim, void *stream) {
    (void)stream;
    return nll_fwd(x, W, bias, target, logits, loss, NULL, stats, workspace, rows, vocab, dim);
}
int fwp_nll_stats_bwd(const float *x, const float *W, const float *logits, const float *stats, const int64_t *target,
                      const float *gloss, float *gx, float *gW, float *gbias, float *workspace, int rows, int vocab, int dim,
                      void *stream) {
    float *d = malloc(sizeof(float) * rows * vocab);
    for (long long r = 0; r < rows; r++)
        for (long long v = 0; v < vocab; v++)
            d[r * vocab + v] = target[r] == -100 ? 0 : target[r] < 0 || target[r] >= vocab ? NAN : (float)((exp(logits[r * vocab + v] - stats[2 * r]) * stats[2 * r + 1] -
                                                            (v == target[r])) * gloss[r]);
    const fwp_mm_epilogue epi = {NULL, NULL, NULL, gbias, 0};
    if (gx) fwp_matmul(FWP_MM_NN, d, vocab, W, dim, gx, dim, rows, dim, vocab, NULL, workspace, stream);
    if (gW) fwp_matmul(FWP_MM_TN, d, vocab, x, dim, gW, dim, vocab, dim, rows, &epi, workspace, stream);
    free(d);
    return 0;
}

int fwp_rows_matmul(const float *x, const float *gamma, const float *beta, float eps, float *y, const float *W,
                    const float *bias, const float *residual, int relu, float *out, int rows, int N, int K, void *stream) {
    float *z = malloc(sizeof(float) * rows * K);
    for (long long r = 0; r < rows; r++)
        if (gamma) norm_row(x + r * K, gamma, beta, z + r * K, NULL, K, eps);
        else memcpy(z + r * K, x + r * K, sizeof(float) * K);
    if (y) memcpy(y, z, sizeof(float) * rows * K);
    const fwp_mm_epilogue epi = {bias, residual, NULL, NULL, relu};
    fwp_matmul(FWP_MM_NT, z, K, W, K, out, N, rows, N, K, &epi, NULL, stream);
    free(z);
    return 0;
}
int fwp_deltanet_step(const float *qkvb, const float *from, float *to, float *out, int B, int H, int D, float q_scale,
                      void *stream) {
    (void)stream;
    g_calls++;
    const long long R = (long long)B * H, S = R * D * D;
    const double s = sum_flat(qkvb, R * (3 * D + 1)) + q_scale;
    for (long long i = 0; i < S; i++) to[i] = (from ? from[i] : 0) + 1.0f;
    fill(out, R * D, s);
    return 0;
}
int fwp_embed(const float *table, const int64_t *ids, const float *inv_freq, float *out, int T, int B, int d,
              long long n_token, float scale, float clamp, void *stream) {
    (void)stream;
    g_calls++;
    for (long long r = 0; r < (long long)T * B; r++)
        for (int j = 0; j < d; j++) {
            double pos = T - 1 - r / B;
            if (clamp > 0 && pos > clamp) pos = clamp;
            const double phase = pos * inv_freq[j % (d / 2)];
            const float e = ids[r] >= 0 && ids[r] < n_token ? table[ids[r] * d + j] : NAN;
            out[r * d + j] = (float)(e * scale + (j < d / 2 ? sin(phase) : cos(phase)));
        }
    return 0;
}
