// Register-state kernels of the Recurrent Delta Net op (rec_update_fwm_tanh) for D in {16, 32}.
//
// On top of the delta-rule state, the slow recurrent matrices R_q, R_k, R_v of the head are held
// in VGPRs in the same layout as the state; the gradients of R_* are accumulated by a wave of their own on the matrix
// cores and written out once per sequence.  16 x 16: a step on one wave, the fed-back vector tanh(out_{t-1}) and the
// activated q and k "grouped" (every lane of group m holds entry m), periodic operands through ds_bpermute, the softmax
// maxima/sums, the beta logit and the softmax-Jacobian dot products as wave-wide reductions.  32 x 32: vectors in half and
// pair form (fwp_reg.hpp), two waves to a sequence forward and four backward (few steps of many sequences: two, as 16 x 16).  512 sequences of 256 steps, against the
// former's kernels for 32 x 32: forward 144 -> 120 us, backward with its sum over the sequences 197 -> 131 us.  Matrices come and go by way of LDS (see
// forms::Matrix): of 20 steps, 512 / 1024 / 2048 sequences, forward 19.3 / 30.1 / 52.6 -> 12.9 / 15.2 / 23.4 us, backward 23.9 / 41.1 / 75.0 -> 23.1 / 39.5 / 71.8.
#include "fwp_reg.hpp"
#include "fwp_mfma.hpp"

namespace fwp {
namespace {

__device__ __forceinline__ float fast_tanh(float x) {
    return 1.f - fast_div(2.f, 1.f + __expf(2.f * x));
}
__device__ __forceinline__ float fast_sigmoid(float x) {
    return fast_div(1.f, 1.f + __expf(-x));
}

// ------------------------------------------------------------------ forward

struct RecFwdOps {
    float qx, kx, vx, bx;
};

template <int RING, int PF, int WPB>
__global__ __launch_bounds__(kWave * WPB) void k_rec_fwd_reg(
    fwp_view qx, fwp_view kx, fwp_view vx, fwp_view bx, const float *__restrict__ Rq,
    const float *__restrict__ Rk, const float *__restrict__ Rv, const float *__restrict__ rb,
    float *__restrict__ W, float *__restrict__ hstate, float *__restrict__ out,
    float *__restrict__ q_act, float *__restrict__ k_act, float *__restrict__ beta_act,
    float *__restrict__ vdiff, float *__restrict__ ckpt, int H, int L, int chunk, int nchunk,
    int nseq) {
    constexpr int D = 16;
    using G = Geo<D>;
    constexpr int S = G::S, R = G::R, NP = G::NP;
    static_assert(kTile % RING == 0 && PF < RING, "ring must divide the tile");
    __shared__ __align__(16) float sq_[WPB][2][kTile * D];
    __shared__ __align__(16) float sk_[WPB][2][kTile * D];
    __shared__ __align__(16) float sv_[WPB][2][kTile * D];
    __shared__ __align__(16) float sb_[WPB][2][kTile];
    __shared__ __align__(16) float sout_[WPB][4][kTile * D + 16];   // staged out, vdiff, q, k tiles
    __shared__ __align__(16) float sba_[WPB][kTile];                // staged beta after the sigmoid

    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);   // uniform: lets the compiler branch on it in scalar code
    const int lane = threadIdx.x % kWave, col = lane / S, sl = lane % S, per = lane % 16;
    const int64_t seq = (int64_t)blockIdx.x * WPB + wave;
    if (seq >= nseq) return;
    const int n = (int)(seq / H), h = (int)(seq % H);
    auto &sq = sq_[wave];
    auto &sk = sk_[wave];
    auto &sv = sv_[wave];
    auto &sb = sb_[wave];
    auto &sout = sout_[wave];
    auto &sba = sba_[wave];
    const float *qb = row(qx, n, h, 0), *kb = row(kx, n, h, 0), *vb = row(vx, n, h, 0),
                *bb = row(bx, n, h, 0);

    // column `col` of the state and of the head's three recurrent matrices
    float Wc[R], Rqc[R], Rkc[R], Rvc[R];
#pragma unroll
    for (int jj = 0; jj < R; jj++) {
        const int e = reg_index<D>(lane, jj);
        Wc[jj] = W[(seq * D + e) * D + col];
        Rqc[jj] = Rq[((int64_t)h * D + e) * D + col];
        Rkc[jj] = Rk[((int64_t)h * D + e) * D + col];
        Rvc[jj] = Rv[((int64_t)h * D + e) * D + col];
    }
    const float rb_m = rb[(int64_t)h * D + col];
    float hcur = hstate[seq * D + col];

    TileRegs<D> pq, pk, pv;
    float pb = 0.f;
    const int lrow = lane / (D / 4), lc4 = lane % (D / 4);
    const float *qlane = qb + lrow * qx.sL + 4 * lc4, *klane = kb + lrow * kx.sL + 4 * lc4,
                *vlane = vb + lrow * vx.sL + 4 * lc4;
    auto fetch = [&](int t0) {
        if (t0 + kTile <= L) {
            pq.template fetch<true>(qlane, qx.sL, t0, L, lane);
            pk.template fetch<true>(klane, kx.sL, t0, L, lane);
            pv.template fetch<true>(vlane, vx.sL, t0, L, lane);
        } else {
            pq.template fetch<false>(qlane, qx.sL, t0, L, lane);
            pk.template fetch<false>(klane, kx.sL, t0, L, lane);
            pv.template fetch<false>(vlane, vx.sL, t0, L, lane);
        }
        pb = bb[(int64_t)min(t0 + per, L - 1) * bx.sL];
    };
    auto commit = [&](int buf) {
        pq.commit(sq[buf], lane);
        pk.commit(sk[buf], lane);
        pv.commit(sv[buf], lane);
        sb[buf][per] = pb;
    };

    float *stage = sout[sl] + col;                       // one LDS write per step: s = 0..3 -> out, vdiff, q, k
    const bool save = vdiff != nullptr;
    float *out_rows = out + seq * L * D;
    auto flush = [&](int t0) {
        flush_tile<D>(sout[0], out_rows, t0, L, lane);
        if (save) {
            flush_tile<D>(sout[1], vdiff + seq * L * D, t0, L, lane);
            flush_tile<D>(sout[2], q_act + seq * L * D, t0, L, lane);
            flush_tile<D>(sout[3], k_act + seq * L * D, t0, L, lane);
            const float b = sba[per];
            if (lane < kTile && t0 + lane < L) beta_act[seq * L + t0 + lane] = b;
        }
    };

    auto load_ops = [&](RecFwdOps &o, int buf, int tt) {
        o.qx = sq[buf][tt * D + col];
        o.kx = sk[buf][tt * D + col];
        o.vx = sv[buf][tt * D + col];
        o.bx = sb[buf][tt];
    };
    auto compute = [&](const RecFwdOps &o, int tt) {
        const float y_m = fast_tanh(hcur);
        float y[NP], kp[NP], qp[NP];
        to_periodic<D>(y_m, y, lane);
        // (needs no periodic operand: runs while the conversion above is on its way)
        const float b = pinned(fast_sigmoid(o.bx + across_groups<S>(rb_m * y_m, OpSum())));
        const float qa = o.qx + group_sum<S>(dot_rot<D>(Rqc, y));
        const float ka = o.kx + group_sum<S>(dot_rot<D>(Rkc, y));
        const float va = o.vx + group_sum<S>(dot_rot<D>(Rvc, y));
        const float eq = __expf(softmax_shifted<S>(qa));
        const float ek = __expf(softmax_shifted<S>(ka));
        // The softmaxes are eq / sum(eq) and ek / sum(ek); the state is read and written with eq and
        // ek and the results are scaled afterwards: the wave-wide sums then run beside the reads
        // instead of ahead of them on the sequential path.
        to_periodic<D>(ek, kp, lane);
        to_periodic<D>(eq, qp, lane);
        const float rk = fast_div(1.f, across_groups<S>(ek, OpSum()));
        const float rq = fast_div(1.f, across_groups<S>(eq, OpSum()));
        const float d = fmaf(-group_sum<S>(dot_rot<D>(Wc, kp)), rk, va);
        rank1_rot<D>(Wc, kp, b * d * rk);
        hcur = group_sum<S>(dot_rot<D>(Wc, qp)) * rq;
        hcur = pinned(hcur);
        const float o_d = pinned(d), o_q = pinned(eq * rq), o_k = pinned(ek * rk);
        stage[tt * D] = sl == 0 ? hcur : (sl == 1 ? o_d : (sl == 2 ? o_q : o_k));
        sba[tt] = b;
    };

    const int ntile = (L + kTile - 1) / kTile;
    fetch(0);
    commit(0);
    if (ntile > 1) fetch(kTile);
    RecFwdOps ring[RING];
#pragma unroll
    for (int p = 0; p < PF; p++) load_ops(ring[p], 0, p);

    for (int it = 0; it < ntile; it++) {
        const int buf = it & 1, t0 = it * kTile;
        const int nst = min(kTile, L - t0);
        if (it + 1 < ntile) commit(buf ^ 1);
        if (it > 0) flush(t0 - kTile);
        if (it + 2 < ntile) fetch(t0 + 2 * kTile);
        if (nst == kTile) {
#pragma unroll
            for (int tt = 0; tt < kTile; tt++) {
                const int nt = tt + PF;
                if (nt < kTile) load_ops(ring[nt % RING], buf, nt);
                else load_ops(ring[nt % RING], buf ^ 1, nt - kTile);
                compute(ring[tt % RING], tt);
            }
        } else {  // ragged last tile: not pipelined
            for (int tt = 0; tt < nst; tt++) {
                RecFwdOps o;
                load_ops(o, buf, tt);
                compute(o, tt);
            }
        }
        const int t_end = t0 + nst;
        if (ckpt && (t_end % chunk == 0 || t_end == L)) {
            float *c = ckpt + (seq * nchunk + (t_end - 1) / chunk) * D * D;
#pragma unroll
            for (int jj = 0; jj < R; jj++) c[reg_index<D>(lane, jj) * D + col] = Wc[jj];
        }
    }
    flush((ntile - 1) * kTile);
#pragma unroll
    for (int jj = 0; jj < R; jj++) W[(seq * D + reg_index<D>(lane, jj)) * D + col] = Wc[jj];
    if (sl == 0) hstate[seq * D + col] = hcur;
}

// ------------------------------------------- forward, 32 x 32 states, two waves per sequence
//
// Wave S carries the steps; wave T, one tile ahead and behind, loads the inputs and stores the results, a tenth of the
// instructions that were the sequential wave's.  No product needs a conversion of its operand: R_q and R_k take tanh(h) in pair form and
// give q and k in half form, one in each half of the wave (one exponential, one sum for both softmaxes), which the state takes to give
// v_old and h in pair form.  What bounds it: the wave's own instructions, about 160 vector ones of 220 a step, 30 of
// them wait states, in 1070 cycles.
// The softmaxes' shift costs no step anything: T takes a row's largest entry off qx and kx, and what R adds to it is below the sum of a
// column of |R| (|tanh| <= 1).  Where that is beyond kFar the largest of the sums is looked for in each step.
// Steps to a tile: 8 take 15 KB a sequence, so that eight fit a CU
constexpr int kFwdTile = 8;
struct RecFwdTile {
    float qk[kFwdTile * 64], v[kFwdTile * 32], b[kFwdTile];      // qx and kx; vx; bx
    float act[kFwdTile * 64];                              // the softmaxes
    float hd[kFwdTile * 64];                               // by 16: entries 0..15 of h, of v - v_old, 16..31 of either
    float ba[kFwdTile];                                    // beta
};
typedef RecFwdTile RecFwdLds[2];
static_assert(sizeof(RecFwdTile) >= 4096, "a matrix on its way");

struct RecFwdArgs {
    fwp_view qx, kx, vx, bx;
    const float *Rq, *Rk, *Rv, *rb;
    float *W, *h, *out, *q_act, *k_act, *beta_act, *vdiff, *ckpt;
    int H, L, chunk, nchunk, nseq;
};

struct RecFwdOps2 {
    float qk, v, b;
};

__device__ __forceinline__ void rec_fwd_steps(RecFwdLds &M, const RecFwdArgs &g, int64_t seq, int lane) {
    using namespace forms;
    constexpr float kFar = 20.f;
    const int half = forms::half(lane), pair = forms::pair(lane), hd = (int)(seq % g.H), L = g.L;
    float W[16], Rq[16], Rk[16], Rv[16], far = 0.f, far_k = 0.f;
    {
        // through the second tile's place, which the other wave fills from its first step on
        float *const stage = reinterpret_cast<float *>(&M[1]);
        const int64_t R = (int64_t)hd * 1024;
        Matrix a, b;
        a.fetch(g.Rq + R, lane), b.fetch(g.Rk + R, lane);
        a.put(stage, lane);
#pragma unroll
        for (int j = 0; j < 16; j++) Rq[j] = stage[terms_of_half(lane, j) * 32 + half];
        a.fetch(g.Rv + R, lane);
        b.put(stage, lane);
#pragma unroll
        for (int j = 0; j < 16; j++) Rk[j] = stage[terms_of_half(lane, j) * 32 + half];
        b.fetch(g.W + seq * 1024, lane);
        a.put(stage, lane);
#pragma unroll
        for (int j = 0; j < 16; j++) Rv[j] = stage[terms_of_half(lane, j) * 32 + half];
        b.put(stage, lane);
#pragma unroll
        for (int j = 0; j < 16; j++) W[j] = stage[terms_of_pair(lane, j) * 32 + pair];
    }
#pragma unroll
    for (int j = 0; j < 16; j++) far += fabsf(Rq[j]), far_k += fabsf(Rk[j]);
    const bool near = !__any(!(sum_to_half(far) <= kFar) || !(sum_to_half(far_k) <= kFar));
    const float rb = g.rb[hd * 32 + pair];
    float h = g.h[seq * 32 + pair];
    const bool first = lane % 32 < 16;

    // where this lane reads and writes in a tile's rows
    const float *qk_at, *v_at, *b_at;
    float *out_at, *ba_at;
    int zero = 0;
    asm volatile("" : "+v"(zero));      // addresses that are the same in all lanes stay in vector registers
    const auto load_ops = [&](RecFwdOps2 &o, int tt) {
        o.qk = qk_at[tt * 64], o.v = v_at[tt * 32], o.b = b_at[tt];
    };
    const auto step = [&](const RecFwdOps2 &o, int tt) __attribute__((always_inline)) {
        const float y = ready(fast_tanh(h));
        float q, k, v;
        dot3(Rq, Rk, Rv, y, q, k, v);
        swap32(q, k);
        float x = (q + k) + o.qk;
        if (__builtin_expect(!near, 0)) {
            OpMax op;
            float m = op(x, dpp<kQuadXor1>(x));
            m = op(m, dpp<kQuadXor2>(m));
            m = op(m, dpp<0x141>(m));
            m = op(m, dpp<0x140>(m));
            float n = m;
            swap16(m, n);
            x -= op(m, n);
        }
        // the softmaxes are e / sum(e): the state is read and written with e, and results are scaled afterwards
        const float e = __expf(x);
        q = k = e;
        swap32(q, k);
        ready(q, k);
        const float r = fast_div(1.f, sums_of_halves(e));
        v = half_shares_to_pair(v) + o.v;
        const float rq = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, r), 0)),
                    rk = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, r), 32));
        const float b = fast_sigmoid(o.b + sum_of_pair(rb * y));
        const float d = fmaf(-sum_to_pair(dot(W, k)), rk, v);
        rank1(W, k, b * d * rk);
        h = sum_to_pair(dot(W, q)) * rq;
        const float o_h = pinned(h), o_d = pinned(d);
        out_at[tt * 64] = e * r;
        out_at[kFwdTile * 64 + tt * 64] = first ? o_h : o_d;
        ba_at[tt] = b;
    };

    const int ntile = (L + kFwdTile - 1) / kFwdTile;
    lds_barrier();
    for (int it = 0; it < ntile; it++) {
        RecFwdTile &T = M[it & 1];
        qk_at = T.qk + lane, v_at = T.v + pair, b_at = T.b + zero, out_at = T.act + lane, ba_at = T.ba + zero;
        const int nst = min(kFwdTile, L - it * kFwdTile);
        if (nst == kFwdTile) {
            RecFwdOps2 ring[2];
            load_ops(ring[0], 0);
#pragma unroll
            for (int tt = 0; tt < kFwdTile; tt++) {
                if (tt + 1 < kFwdTile) load_ops(ring[(tt + 1) & 1], tt + 1);
                step(ring[tt & 1], tt);
            }
        } else {
#pragma unroll 1
            for (int tt = 0; tt < nst; tt++) {
                RecFwdOps2 o;
                load_ops(o, tt);
                step(o, tt);
            }
        }
        const int t_end = it * kFwdTile + nst;
        if (g.ckpt && t_end % g.chunk == 0 && t_end < L) {
            float *c = g.ckpt + (seq * g.nchunk + t_end / g.chunk - 1) * 1024;
#pragma unroll
            for (int j = 0; j < 16; j++) c[terms_of_pair(lane, j) * 32 + pair] = W[j];
        }
        lds_barrier();
    }
    // through the last tile but one's place, which the other wave has read
    float *const stage = reinterpret_cast<float *>(&M[ntile & 1]);
    Matrix last;
#pragma unroll
    for (int j = 0; j < 16; j++) stage[terms_of_pair(lane, j) * 32 + pair] = W[j];
    last.take(stage, lane);
    last.store(g.W + seq * 1024, lane);
    if (g.ckpt) last.store(g.ckpt + (seq * g.nchunk + g.nchunk - 1) * 1024, lane);
    if (first) g.h[seq * 32 + pair] = h;
}

__device__ __forceinline__ void rec_fwd_tiles(RecFwdLds &M, const RecFwdArgs &g, int64_t seq, int lane) {
    constexpr int D = 32, NV4 = Geo<D, kFwdTile>::NV4;
    const int n = (int)(seq / g.H), hd = (int)(seq % g.H), L = g.L, row8 = lane / 8, c4 = lane % 8, per = lane % kFwdTile;
    const float *q = row(g.qx, n, hd, 0) + row8 * g.qx.sL + 4 * c4, *k = row(g.kx, n, hd, 0) + row8 * g.kx.sL + 4 * c4,
                *v = row(g.vx, n, hd, 0) + row8 * g.vx.sL + 4 * c4, *b = row(g.bx, n, hd, 0);
    TileRegs<D, kFwdTile> pq, pk, pv;
    float pb = 0.f;
    const auto fetch = [&](int t0) {
        if (t0 + kFwdTile <= L) {
            pq.template fetch<true>(q, g.qx.sL, t0, L, lane);
            pk.template fetch<true>(k, g.kx.sL, t0, L, lane);
            pv.template fetch<true>(v, g.vx.sL, t0, L, lane);
        } else {
            pq.template fetch<false>(q, g.qx.sL, t0, L, lane);
            pk.template fetch<false>(k, g.kx.sL, t0, L, lane);
            pv.template fetch<false>(v, g.vx.sL, t0, L, lane);
        }
        pb = b[(int64_t)min(t0 + per, L - 1) * g.bx.sL];
    };
    const auto less_largest = [&](float4 x) {
        const float m = row_reduce<D>(OpMax()(OpMax()(x.x, x.y), OpMax()(x.z, x.w)), OpMax());
        return make_float4(x.x - m, x.y - m, x.z - m, x.w - m);
    };
    const auto commit = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NV4; i++) {
            float *to = M[buf].qk + (row8 + 8 * i) * 64 + 4 * c4;
            *reinterpret_cast<float4 *>(to) = less_largest(pq.r[i]);
            *reinterpret_cast<float4 *>(to + 32) = less_largest(pk.r[i]);
        }
        pv.commit(M[buf].v, lane);
        M[buf].b[per] = pb;
    };
    const int at = c4 < 4 ? 4 * c4 : 16 + 4 * c4;      // of four entries of h in a row of hd
    const auto flush = [&](int it) {
        const int buf = it & 1;
#pragma unroll
        for (int i = 0; i < NV4; i++) {
            const int tt = row8 + 8 * i, t = it * kFwdTile + tt;
            const float4 *hd4 = reinterpret_cast<const float4 *>(M[buf].hd + tt * 64 + at),
                         *a4 = reinterpret_cast<const float4 *>(M[buf].act + tt * 64 + 4 * c4);
            if (t >= L) continue;
            const int64_t to = (seq * L + t) * D + 4 * c4;
            *reinterpret_cast<float4 *>(g.out + to) = hd4[0];
            if (g.vdiff) {
                *reinterpret_cast<float4 *>(g.vdiff + to) = hd4[4];
                *reinterpret_cast<float4 *>(g.q_act + to) = a4[0];
                *reinterpret_cast<float4 *>(g.k_act + to) = a4[8];
            }
        }
        if (g.vdiff && lane < kFwdTile && it * kFwdTile + lane < L) g.beta_act[seq * L + it * kFwdTile + lane] = M[buf].ba[lane];
    };
    const int ntile = (L + kFwdTile - 1) / kFwdTile;
    fetch(0);
    commit(0);
    if (ntile > 1) fetch(kFwdTile);
    lds_barrier();
    for (int it = 0; it < ntile; it++) {
        if (it + 1 < ntile) commit((it + 1) & 1);
        if (it + 2 < ntile) fetch((it + 2) * kFwdTile);
        if (it > 0) flush(it - 1);
        lds_barrier();
    }
    flush(ntile - 1);
}

// NS sequences to a workgroup: waves 0 .. NS-1 carry the steps.  The waves of a workgroup go to the SIMDs in turn.
template <int NS>
__global__ __launch_bounds__(kWave * 2 * NS) void k_rec_fwd_pair(RecFwdArgs g) {
    __shared__ __align__(16) RecFwdLds lds[NS];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const int64_t seq = (int64_t)blockIdx.x * NS + wave % NS;
    if (seq >= g.nseq) {      // the last workgroup's spare waves only keep the barriers' count
        const int ntile = (g.L + kFwdTile - 1) / kFwdTile;
        for (int it = ntile; it >= 0; it--) lds_barrier();
        return;
    }
    if (wave < NS) rec_fwd_steps(lds[wave % NS], g, seq, lane);
    else rec_fwd_tiles(lds[wave % NS], g, seq, lane);
}

// ----------------------------------------------------------------- backward, two waves per sequence

template <int D>
struct RecBwdOps {
    float q[Geo<D>::NP], k[Geo<D>::NP], u[Geo<D>::NP];
    float q_i, k_i, go_i, d_i, y_i, b;
};

// Nearly all of the backward step is sequential (the gradient reaches h_{t-1} through q, k, v and
// beta alike); what is not is the gradient of the slow recurrent weights, sums over time of
// tanh(h_{t-1}) (x) grad_qx, grad_kx, grad_vx and tanh(h_{t-1}) grad_bx.  A second wave, one tile
// of 16 steps behind, takes those tiles from LDS and accumulates the sums on the matrix cores
// (X^T Y over the 16 steps of a tile).  One workgroup barrier per tile; a workgroup holds two
// sequences.
template <int D>
struct RecPairLds {
    float q[2][kTile * D], k[2][kTile * D], go[2][kTile * D], d[2][kTile * D], u[2][kTile * D];
    float y[3][kTile * D];                    // tanh of the delayed output: ring of three tiles
    float grad[2][3][kTile * D + 16];         // staged gqx, gkx, gvx, by tile parity
    float b[2][kTile], gb[2][kTile];
};

template <int D>
__device__ __forceinline__ void rec_bwd_pair_x(RecPairLds<D> &M, const float *__restrict__ q_act,
                                               const float *__restrict__ k_act,
                                               const float *__restrict__ beta_act,
                                               const float *__restrict__ vdiff,
                                               const float *__restrict__ out,
                                               const float *__restrict__ h_init, fwp_view go,
                                               const float *__restrict__ Rq, const float *__restrict__ Rk,
                                               const float *__restrict__ Rv, const float *__restrict__ rb,
                                               const float *__restrict__ ckpt, float *__restrict__ gqx,
                                               float *__restrict__ gkx, float *__restrict__ gvx,
                                               float *__restrict__ gbx, int H, int L, int chunk, int nchunk,
                                               int64_t seq, int lane) {
    using G = Geo<D>;
    constexpr int S = G::S, R = G::R, NP = G::NP, NV4 = G::NV4;
    const int i = lane / S, sl = lane % S, per = lane % 16;
    const int h = (int)(seq % H), n = (int)(seq / H);
    const float *gob = row(go, n, h, 0);
    const float *qb = q_act + seq * L * D, *kb = k_act + seq * L * D, *db = vdiff + seq * L * D,
                *ob = out + seq * L * D, *hib = h_init + seq * D, *bb = beta_act + seq * L;

    // row i of: the state, its gradient (also column i of it) and the recurrent matrices
    float Wr[R], Gr[R], Gc[R], Wnext[R], Rqr[R], Rkr[R], Rvr[R];
#pragma unroll
    for (int jj = 0; jj < R; jj++) {
        const int m = reg_index<D>(lane, jj);
        Gr[jj] = Gc[jj] = Wr[jj] = 0.f;
        Rqr[jj] = Rq[((int64_t)h * D + i) * D + m];
        Rkr[jj] = Rk[((int64_t)h * D + i) * D + m];
        Rvr[jj] = Rv[((int64_t)h * D + i) * D + m];
    }
    const float rb_i = rb[(int64_t)h * D + i];
    float dh_i = 0.f;

    TileRegs<D> pq, pk, pgo, pd, pu, py;
    float pb = 0.f;
    const int lrow = lane / (D / 4), lc4 = lane % (D / 4);
    const float *qlane = qb + lrow * D + 4 * lc4, *klane = kb + lrow * D + 4 * lc4,
                *dlane = db + lrow * D + 4 * lc4, *golane = gob + lrow * go.sL + 4 * lc4;
    auto fetch = [&](int t0) {
        if (t0 + kTile <= L) {
            pq.template fetch<true>(qlane, D, t0, L, lane);
            pk.template fetch<true>(klane, D, t0, L, lane);
            pd.template fetch<true>(dlane, D, t0, L, lane);
            pgo.template fetch<true>(golane, go.sL, t0, L, lane);
        } else {
            pq.template fetch<false>(qlane, D, t0, L, lane);
            pk.template fetch<false>(klane, D, t0, L, lane);
            pd.template fetch<false>(dlane, D, t0, L, lane);
            pgo.template fetch<false>(golane, go.sL, t0, L, lane);
        }
        float bs[NV4];
#pragma unroll
        for (int x = 0; x < NV4; x++) {
            const int t = t0 + lrow + TileRegs<D>::kRowsPerLoad * x;
            bs[x] = bb[min(t, L - 1)];
            // row t of the delayed output is out[t-1], or the initial state for t = 0
            const float *src = t == 0 ? hib + 4 * lc4 : ob + (int64_t)(min(t, L) - 1) * D + 4 * lc4;
            py.r[x] = *reinterpret_cast<const float4 *>(src);
        }
        pu = pd;
        pu.scale_rows(bs);
        pb = bb[min(t0 + per, L - 1)];
    };
    auto commit = [&](int it) {
        const int buf = it & 1;
        pq.commit(M.q[buf], lane);
        pk.commit(M.k[buf], lane);
        pgo.commit(M.go[buf], lane);
        pd.commit(M.d[buf], lane);
        pu.commit(M.u[buf], lane);
        M.b[buf][per] = pb;
#pragma unroll
        for (int x = 0; x < NV4; x++) {
            float4 &r = py.r[x];
            r.x = fast_tanh(r.x); r.y = fast_tanh(r.y); r.z = fast_tanh(r.z); r.w = fast_tanh(r.w);
        }
        py.commit(M.y[it % 3], lane);
    };
    auto fetch_state = [&](int c) {
        const float *src = ckpt + ((seq * nchunk + c) * D + i) * D;
#pragma unroll
        for (int jj = 0; jj < R; jj++) Wnext[jj] = src[reg_index<D>(lane, jj)];
    };
    float *gq_rows = gqx + seq * L * D, *gk_rows = gkx + seq * L * D, *gv_rows = gvx + seq * L * D;

    auto load_ops = [&](RecBwdOps<D> &o, int it, int tt) {
        const int buf = it & 1, off = tt * D;
#pragma unroll
        for (int p = 0; p < NP; p++) {
            o.q[p] = M.q[buf][off + 16 * p + per];
            o.k[p] = M.k[buf][off + 16 * p + per];
            o.u[p] = M.u[buf][off + 16 * p + per];
        }
        o.q_i = M.q[buf][off + i];
        o.k_i = M.k[buf][off + i];
        o.go_i = M.go[buf][off + i];
        o.d_i = M.d[buf][off + i];
        o.y_i = M.y[it % 3][off + i];
        o.b = M.b[buf][tt];
    };
    auto compute = [&](const RecBwdOps<D> &o, int it, int tt) {
        const float g_i = dh_i + o.go_i;                      // gradient of out_t
        float g[NP], a[NP], gqp[NP], gkp[NP];
        // Every conversion of a grouped vector into a periodic operand (ds_bpermute, 60 cycles before its
        // result can be used) is issued as soon as its input exists, with work that does not need it behind it.
        to_periodic<D>(g_i, g, lane);
        // G' = G + q (x) g (both layouts);  r = G'^T k
        rank1_rot<D>(Gc, o.q, g_i);
        const float r_i = group_sum<S>(dot_rot<D>(Gc, o.k));
        const float gvx_i = o.b * r_i;
        const float a_i = -gvx_i;                             // gradient w.r.t. v_old
        to_periodic<D>(a_i, a, lane);
        // gradient of q (after softmax) = W_t g, then through the softmax
        const float dq_i = group_sum<S>(dot_rot<D>(Wr, g));
        const float gqx_i = o.q_i * (dq_i - across_groups<S>(dq_i * o.q_i, OpSum()));
        to_periodic<D>(gqx_i, gqp, lane);
        const float gb = across_groups<S>(r_i * o.d_i, OpSum());
        const float gbx_t = gb * o.b * (1.f - o.b);           // through the sigmoid
        rank1_rot<D>(Gr, g, o.q_i);
        rank1_rot<D, true>(Wr, o.u, o.k_i);                   // W_{t-1}
        rank1_rot<D>(Gc, o.k, a_i);
        float dk_i = dot_rot<D>(Gr, o.u);                     // G' u + W_{t-1} a
        dk_i = group_sum<S>(dot_rot<D>(Wr, a, dk_i));
        rank1_rot<D>(Gr, a, o.k_i);
        // back through the slow recurrent weights to tanh(out_{t-1}) and to out_{t-1}: the terms of q and v
        // (grad_vx = -a, already periodic) while grad_kx is still on its way
        float acc = dot_rot<D>(Rqr, gqp) - dot_rot<D>(Rvr, a);
        const float gkx_i = o.k_i * (dk_i - across_groups<S>(dk_i * o.k_i, OpSum()));
        to_periodic<D>(gkx_i, gkp, lane);
        acc = group_sum<S>(dot_rot<D>(Rkr, gkp, acc));
        acc = fmaf(rb_i, gbx_t, acc);
        dh_i = (1.f - o.y_i * o.y_i) * acc;
        const float o_q = pinned(gqx_i), o_k = pinned(gkx_i), o_v = pinned(gvx_i);
        float *g0 = M.grad[it & 1][0] + tt * D + i, *g1 = M.grad[it & 1][1] + tt * D + i,
              *g2 = M.grad[it & 1][2] + tt * D + i;
        if constexpr (S == 4) {
            *(sl == 0 ? g0 : (sl == 1 ? g1 : g2)) = sl == 0 ? o_q : (sl == 1 ? o_k : o_v);
        } else {
            *(sl == 0 ? g0 : g1) = sl == 0 ? o_q : o_k;
            *g2 = o_v;
        }
        M.gb[it & 1][tt] = gbx_t;
    };
    auto flush = [&](int it) {
        const int t0 = it * kTile;
        flush_tile<D>(M.grad[it & 1][0], gq_rows, t0, L, lane);
        flush_tile<D>(M.grad[it & 1][1], gk_rows, t0, L, lane);
        flush_tile<D>(M.grad[it & 1][2], gv_rows, t0, L, lane);
        const float x = M.gb[it & 1][per];
        if (lane < kTile && t0 + lane < L) gbx[seq * L + t0 + lane] = x;
    };

    const int ntile = (L + kTile - 1) / kTile;
    fetch((ntile - 1) * kTile);
    commit(ntile - 1);
    fetch_state(nchunk - 1);
    if (ntile > 1) fetch((ntile - 2) * kTile);
    __syncthreads();

    for (int it = ntile - 1; it >= 0; it--) {
        const int t0 = it * kTile;
        const int nst = min(kTile, L - t0);
        const int t_end = t0 + nst;
        if (t_end % chunk == 0 || t_end == L) {  // first tile (in reverse) of a chunk: re-anchor W
#pragma unroll
            for (int jj = 0; jj < R; jj++) Wr[jj] = Wnext[jj];
        }
        if (it >= 1) commit(it - 1);
        if (it + 1 < ntile) flush(it + 1);
        if (it >= 1 && t0 % chunk == 0) fetch_state(t0 / chunk - 1);
        if (it >= 2) fetch(t0 - 2 * kTile);
        if (nst == kTile) {
            RecBwdOps<D> ring[2];
            load_ops(ring[(kTile - 1) & 1], it, kTile - 1);
#pragma unroll
            for (int tt = kTile - 1; tt >= 0; tt--) {
                if (tt > 0) load_ops(ring[(tt - 1) & 1], it, tt - 1);
                compute(ring[tt & 1], it, tt);
            }
        } else {  // ragged last tile (first in reverse): not pipelined
            for (int tt = nst - 1; tt >= 0; tt--) {
                RecBwdOps<D> o;
                load_ops(o, it, tt);
                compute(o, it, tt);
            }
        }
        __syncthreads();
    }
    flush(0);
}

typedef float rec_v4f __attribute__((ext_vector_type(4)));

template <int D>
__device__ __forceinline__ void rec_bwd_pair_y(RecPairLds<D> &M, float *__restrict__ workspace, int L,
                                               int64_t seq, int lane) {
    constexpr int NT = D / 16;
    // acc[x][mt][nt]: lane l, register r holds entry (16 mt + 4 (l / 16) + r, 16 nt + l % 16) of
    // sum_t y_t (x) grad_x; accb the same for y_t grad_bx in column 0
    rec_v4f acc[3][NT][NT], accb[NT];
#pragma unroll
    for (int mt = 0; mt < NT; mt++) {
        accb[mt] = rec_v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < 3; x++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) acc[x][mt][nt] = rec_v4f{0.f, 0.f, 0.f, 0.f};
    }
    const int r4 = lane / 16, c = lane % 16;
    auto run_tile = [&](int ty) {
        const int nst = min(kTile, L - ty * kTile);
        const float *y = M.y[ty % 3];
#pragma unroll
        for (int j = 0; j < kTile / 4; j++) {       // four steps to an MFMA: step 4 j + l / 16
            const int tt = 4 * j + r4;
            const bool ok = tt < nst;
            float a[NT], b[3][NT];
#pragma unroll
            for (int mt = 0; mt < NT; mt++) a[mt] = ok ? y[tt * D + 16 * mt + c] : 0.f;
#pragma unroll
            for (int x = 0; x < 3; x++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) b[x][nt] = ok ? M.grad[ty & 1][x][tt * D + 16 * nt + c] : 0.f;
            const float bcol = ok && c == 0 ? M.gb[ty & 1][tt] : 0.f;
#pragma unroll
            for (int mt = 0; mt < NT; mt++) {
#pragma unroll
                for (int x = 0; x < 3; x++)
#pragma unroll
                    for (int nt = 0; nt < NT; nt++)
                        acc[x][mt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[mt], b[x][nt], acc[x][mt][nt], 0, 0, 0);
                accb[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[mt], bcol, accb[mt], 0, 0, 0);
            }
        }
    };
    const int ntile = (L + kTile - 1) / kTile;
    __syncthreads();
    for (int it = ntile - 1; it >= 0; it--) {     // the tile X works on; this wave is one behind
        if (it + 1 < ntile) run_tile(it + 1);
        __syncthreads();
    }
    run_tile(0);
    // this sequence's share of the parameter gradients: [gRq | gRk | gRv | grb], rows e, columns m
    float *ws = workspace + seq * (3 * D * D + D);
#pragma unroll
    for (int mt = 0; mt < NT; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int e = 16 * mt + 4 * r4 + r;
#pragma unroll
            for (int x = 0; x < 3; x++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++) ws[x * D * D + e * D + 16 * nt + c] = acc[x][mt][nt][r];
            if (c == 0) ws[3 * D * D + e] = accb[mt][r];
        }
}

// NS sequences to a workgroup: waves 0 .. NS-1 carry the steps, waves NS .. 2 NS - 1 the sums.  The waves
// of a workgroup go to the SIMDs in turn; with four sequences each SIMD of the CU gets one wave of
// either kind, whereas two workgroups of two sequences on a CU both put their heavy waves on the same
// two SIMDs.
template <int D, int NS>
__global__ __launch_bounds__(kWave * 2 * NS) void k_rec_bwd_pair(
    const float *__restrict__ q_act, const float *__restrict__ k_act,
    const float *__restrict__ beta_act, const float *__restrict__ vdiff,
    const float *__restrict__ out, const float *__restrict__ h_init, fwp_view go,
    const float *__restrict__ Rq, const float *__restrict__ Rk, const float *__restrict__ Rv,
    const float *__restrict__ rb, const float *__restrict__ ckpt, float *__restrict__ gqx,
    float *__restrict__ gkx, float *__restrict__ gvx, float *__restrict__ gbx,
    float *__restrict__ workspace, int H, int L, int chunk, int nchunk, int nseq) {
    extern __shared__ __align__(16) unsigned char pair_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const int64_t seq = (int64_t)blockIdx.x * NS + wave % NS;
    RecPairLds<D> &M = reinterpret_cast<RecPairLds<D> *>(pair_lds)[wave % NS];
    if (seq >= nseq) {   // the last workgroup's spare waves only keep the barriers' count
        const int ntile = (L + kTile - 1) / kTile;
        for (int it = ntile; it >= 0; it--) __syncthreads();
        return;
    }
    if (wave < NS)
        rec_bwd_pair_x<D>(M, q_act, k_act, beta_act, vdiff, out, h_init, go, Rq, Rk, Rv, rb, ckpt, gqx, gkx, gvx,
                          gbx, H, L, chunk, nchunk, seq, lane);
    else
        rec_bwd_pair_y<D>(M, workspace, L, seq, lane);
}

// ------------------------------------------- backward, 32 x 32 states, four waves per sequence
//
// What the gradient of h_t has to pass through is W_{t-1} g, two softmaxes and R; the rest of the step is linear in it and is
// prepared beside.  With g the gradient of h_t, G that of the state after step t, W the state before it, u = b (v - v_old), P = G^T k
// and Q = G u:
//   grad_vx = b (P + (q.k) g), a = -grad_vx,   grad_bx = b (1 - b) (P.d + (q.k) (g.d)),
//   grad_q = W g + (g.u) k,   grad_k = Q + (g.u) q + W a,   W a = -b (W P + (q.k) W g),
// so of the matrices only W and R meet the step's own vectors.  Wave X carries that; wave C keeps G by columns and a state of its own
// and prepares P, P.d and W P of the next step, wave D keeps G by rows and prepares its Q, each from the g that X hands over right at the
// start of a step: one barrier a step.  Wave Y loads and stores, a sixteenth of a tile's work in each step, and sums the
// gradients of R on the matrix cores.  X is what bounds it: 180 instructions a step (134 vector ones, 22 wait states), where one wave that forms everything in turn takes about 200, most of
// them one behind the other.
// No product's operand is converted (see forms): g and P in pair form, q and k in half form, of which X holds q in one half of
// the wave and k in the other for both softmaxes at once; the two products with R_q and R_k are one of 64 terms.
struct RecBwdTile {
    float qk[kTile * 64], u[kTile * 32], d[kTile * 32], go[kTile * 32], dt[kTile * 32];      // dt: 1 - tanh(h_{t-1})^2
    float4 sc[kTile];           // b, q.k, b (1 - b)
    float co[kTile * 2];        // 1, -b q.k
    float gqk[kTile * 64], gv[kTile * 32], gb[kTile];
};
struct RecBwdLds {
    RecBwdTile tile[2];
    float y[3][kTile * 32];     // tanh(h_{t-1}): a ring of three tiles
    // from step to step, by its parity; the first halves of Q and WP stay zero
    float g[2][32], P[2][32], Q[2][64], WP[2][64], Pd[2];
};

// Steps to an iteration of the waves' loops.  All four run at once, each through its own: unrolled by 16 they were 56 KB of
// instructions, as much as the cache that two CUs share holds.
constexpr int kUnroll = 4;

struct RecBwdArgs {
    const float *q_act, *k_act, *beta_act, *vdiff, *out, *h_init;
    fwp_view go;
    const float *Rq, *Rk, *Rv, *rb, *ckpt;
    float *gqx, *gkx, *gvx, *gbx, *workspace;
    int H, L, chunk, nchunk;
};

struct RecBwdOpsX {
    float pq, pk, k, u, d, go, dt, co;      // q beside k, k beside q, k
    float4 sc;
};

// The state after step t of a chunk that ends there, as its rows (results of a product over the values in half form)
__device__ __forceinline__ void rec_state_rows(float (&W)[16], const RecBwdArgs &g, int64_t seq, int c, int lane) {
    const float *src = g.ckpt + ((seq * g.nchunk + c) * 32 + forms::half(lane)) * 32;
#pragma unroll
    for (int j = 0; j < 16; j++) W[j] = src[forms::terms_of_half(lane, j)];
}

__device__ __forceinline__ void rec_bwd_x(RecBwdLds &M, const RecBwdArgs &g, int64_t seq, int lane) {
    using namespace forms;
    const int half = forms::half(lane), pair = forms::pair(lane), hd = (int)(seq % g.H), L = g.L;
    float W[16], Wnext[16], R0[16], R1[16], Rv[16];
    {
        // through where this wave's results of a tile are kept
        static_assert(sizeof(M.tile[0].gqk) == 4096, "a matrix on its way");
        float *const stage = M.tile[0].gqk;
        const int64_t R = (int64_t)hd * 1024;
        // a row of lanes holds half of one vector of (grad_qx, grad_kx): entries lane % 16 and 16 + lane % 16 of the results
        const auto read = [&] {
#pragma unroll
            for (int j = 0; j < 16; j++) R0[j] = stage[lane % 16 * 32 + terms_of_pair(lane, j)], R1[j] = stage[(16 + lane % 16) * 32 + terms_of_pair(lane, j)];
        };
        Matrix a, b, c;
        a.fetch(g.Rq + R, lane), b.fetch(g.Rk + R, lane), c.fetch(g.Rv + R, lane);
        a.put(stage, lane);
        if (lane < 32) read();
        b.put(stage, lane);
        if (lane >= 32) read();
        c.put(stage, lane);
#pragma unroll
        for (int j = 0; j < 16; j++) Rv[j] = stage[half * 32 + terms_of_half(lane, j)], W[j] = 0.f;
    }
    const float rb = g.rb[hd * 32 + pair];
    float dh = 0.f;
#pragma unroll
    for (int j = 0; j < 16; j++) R0[j] = pinned(R0[j]), R1[j] = pinned(R1[j]), Rv[j] = pinned(Rv[j]);      // they are waited for here, not in each step
    const float *qk_at, *kq_at, *k_at, *v_at, *co_at;
    float *gqk_at, *gv_at, *gb_at;
    const float4 *sc_at;
    int zero = 0;
    asm volatile("" : "+v"(zero));
    const auto load_ops = [&](RecBwdOpsX &o, int tt) {
        o.pq = qk_at[tt * 64], o.pk = kq_at[tt * 64], o.k = k_at[tt * 64];
        o.u = v_at[tt * 32], o.d = v_at[kTile * 32 + tt * 32], o.go = v_at[2 * kTile * 32 + tt * 32], o.dt = v_at[3 * kTile * 32 + tt * 32];
        o.sc = sc_at[tt], o.co = co_at[2 * tt];
    };
    // W: before step t.  n: the operands of step t - 1 (more: it is of this tile), for which W is prepared while the sums below are on their way;
    // load(): those of step t - 2
    const auto step = [&](const RecBwdOpsX &o, const RecBwdOpsX &n, int tt, bool more, auto load) __attribute__((always_inline)) {
        const int p = tt & 1;
        const float b = o.sc.x, qk = o.sc.y;
        const float h = dh + o.go;                 // the gradient of h_t
        M.g[p][pair] = h;
        const float z1 = pinned(dot(W, ready(h)));
        lds_barrier();
        const float P = M.P[p][pair], Q = M.Q[p][lane], WP = M.WP[p][lane], Pd = M.Pd[p];
        load();
        const float z = sum_to_half(z1), gd = sum_of_pair(h * o.d);
        if (more) rank1<true>(W, n.u, n.k);
        const float w = fmaf(o.co, z, fmaf(o.pk, b * gd, fmaf(-b, WP, Q)));      // grad_q beside grad_k
        const float gv = ready(b * fmaf(qk, h, P)), gb = o.sc.z * fmaf(qk, gd, Pd);
        // the sums of w q and w k, with R_v grad_vx while their stages wait for one another
        float v[1][4], m = w * o.pq;
        dot_part<0>(Rv, gv, v);
        m += dpp<kQuadXor1>(m);
        dot_part<4>(Rv, gv, v);
        m += dpp<kQuadXor2>(m);
        dot_part<8>(Rv, gv, v);
        m += dpp<0x141>(m);
        dot_part<12>(Rv, gv, v);
        m += dpp<0x140>(m);
        const float a2 = (v[0][0] + v[0][1]) + (v[0][2] + v[0][3]);
        const float gqk = ready(o.pq * (w - sum_to_pair(m)));
        float a0, a1;
        dot2(R0, R1, gqk, a0, a1);
        swap16(a0, a1);
        dh = o.dt * fmaf(rb, gb, half_shares_to_pair((a0 + a1) + a2));
        gqk_at[tt * 64] = gqk, gv_at[tt * 32] = gv, gb_at[tt] = gb;
    };
    const int ntile = (L + kTile - 1) / kTile;
    lds_barrier();
#pragma unroll
    for (int j = 0; j < 16; j++) Wnext[j] = M.tile[1].gqk[half * 32 + terms_of_half(lane, j)];      // the last state, from wave C
    for (int it = ntile - 1; it >= 0; it--) {
        const int t0 = it * kTile, nst = min(kTile, L - t0);
        RecBwdTile &T = M.tile[it & 1];
        qk_at = T.qk + lane, kq_at = T.qk + (lane ^ 32), k_at = T.qk + 32 + half, v_at = T.u + pair, co_at = T.co + lane / 32;
        sc_at = T.sc + zero, gqk_at = T.gqk + lane, gv_at = T.gv + pair, gb_at = T.gb + zero;
        if ((t0 + nst) % g.chunk == 0 || it == ntile - 1)
#pragma unroll
            for (int j = 0; j < 16; j++) W[j] = Wnext[j];
        if (it && t0 % g.chunk == 0) rec_state_rows(Wnext, g, seq, t0 / g.chunk - 1, lane);
        if (nst == kTile) {
            RecBwdOpsX ring[kUnroll];
            load_ops(ring[kUnroll - 1], kTile - 1);
            load_ops(ring[kUnroll - 2], kTile - 2);
            rank1<true>(W, ring[kUnroll - 1].u, ring[kUnroll - 1].k);
#pragma unroll 1
            for (int tb = kTile - kUnroll; tb >= 0; tb -= kUnroll)
#pragma unroll
                for (int j = kUnroll - 1; j >= 0; j--)
                    step(ring[j], ring[(j + kUnroll - 1) % kUnroll], tb + j, j || tb, [&] {
                        if (j >= 2 || tb) load_ops(ring[(j + kUnroll - 2) % kUnroll], tb + j - 2);
                    });
        } else {
#pragma unroll 1
            for (int tt = nst - 1; tt >= 0; tt--) {
                RecBwdOpsX o;
                load_ops(o, tt);
                rank1<true>(W, o.u, o.k);
                step(o, o, tt, false, [] {});
            }
        }
    }
    lds_barrier();
}

// G by columns: P, P.d and W P of step t - 1 from the g of step t
__device__ __forceinline__ void rec_bwd_c(RecBwdLds &M, const RecBwdArgs &g, int64_t seq, int lane) {
    using namespace forms;
    const int half = forms::half(lane), pair = forms::pair(lane), L = g.L, ntile = (L + kTile - 1) / kTile;
    float W[16], Wnext[16], G[16], P = 0.f;
    float *const stage = M.tile[1].gqk;      // wave X reads it too, before it keeps results there
    Matrix last;
    last.fetch(g.ckpt + (seq * g.nchunk + g.nchunk - 1) * 1024, lane);
    last.put(stage, lane);
#pragma unroll
    for (int j = 0; j < 16; j++) W[j] = stage[half * 32 + terms_of_half(lane, j)], G[j] = Wnext[j] = 0.f;
    M.P[0][half] = M.P[1][half] = 0.f;
    M.Q[0][lane] = M.Q[1][lane] = M.WP[0][lane] = M.WP[1][lane] = 0.f;
    M.Pd[0] = M.Pd[1] = 0.f;
    lds_barrier();
    const auto rewind = [&](const RecBwdTile &T, int tt) { rank1<true>(W, T.u[tt * 32 + pair], T.qk[tt * 64 + 32 + half]); };
    rewind(M.tile[(ntile - 1) & 1], (L - 1) & (kTile - 1));
    struct Ops {
        float q, k, k1, u1, d1;
        float4 sc;
    };
    const auto load_ops = [&](Ops &o, const RecBwdTile &T, const RecBwdTile &N, int tt, int nt) {
        o.q = T.qk[tt * 64 + half], o.k = T.qk[tt * 64 + 32 + half], o.sc = T.sc[tt];
        o.k1 = N.qk[nt * 64 + 32 + half], o.u1 = N.u[nt * 32 + pair], o.d1 = N.d[nt * 32 + pair];
    };
    const auto step = [&](const Ops &o, int tt, bool anchor, bool more, auto load) __attribute__((always_inline)) {
        const int p = tt & 1;
        if (anchor)
#pragma unroll
            for (int j = 0; j < 16; j++) W[j] = Wnext[j];
        lds_barrier();
        const float h = M.g[p][pair];
        load();
        if (more) rank1<true>(W, o.u1, o.k1);
        const float a = -o.sc.x * fmaf(o.sc.y, h, P);
        rank1(G, o.q, h);
        rank1(G, o.k, a);
        if (!more) return;
        P = sum_to_pair(dot(G, o.k1));
        M.P[p ^ 1][pair] = P;
        const float wp = sum_to_half(dot(W, ready(P)));
        M.WP[p ^ 1][32 + half] = wp;
        M.Pd[p ^ 1] = sum_of_pair(P * o.d1);
    };
    for (int it = ntile - 1; it >= 0; it--) {
        const int t0 = it * kTile, nst = min(kTile, L - t0);
        const RecBwdTile &T = M.tile[it & 1], &N = M.tile[it & 1 ^ 1];
        const bool anchor = it && t0 % g.chunk == 0;
        if (anchor) rec_state_rows(Wnext, g, seq, t0 / g.chunk - 1, lane);
        if (nst == kTile) {
            Ops ring[2];
            load_ops(ring[(kTile - 1) & 1], T, T, kTile - 1, kTile - 2);
#pragma unroll 1
            for (int tb = kTile - kUnroll; tb >= 0; tb -= kUnroll)
#pragma unroll
                for (int j = kUnroll - 1; j >= 0; j--)
                    step(ring[j & 1], tb + j, j == 0 && !tb && anchor, j || tb || it, [&] {
                        if (j > 1 || (j == 0 && tb)) load_ops(ring[(j + 1) & 1], T, T, tb + j - 1, tb + j - 2);
                        else if (j == 1) load_ops(ring[0], T, tb ? T : N, tb, tb ? tb - 1 : kTile - 1);
                    });
        } else {
#pragma unroll 1
            for (int tt = nst - 1; tt >= 0; tt--) {
                Ops o;
                load_ops(o, T, tt ? T : N, tt, tt ? tt - 1 : kTile - 1);
                step(o, tt, tt == 0 && anchor, tt > 0 || it > 0, [] {});
            }
        }
    }
    lds_barrier();
}

// G by rows: Q of step t - 1
__device__ __forceinline__ void rec_bwd_d(RecBwdLds &M, const RecBwdArgs &g, int64_t seq, int lane) {
    using namespace forms;
    const int half = forms::half(lane), pair = forms::pair(lane), L = g.L, ntile = (L + kTile - 1) / kTile;
    float G[16];
#pragma unroll
    for (int j = 0; j < 16; j++) G[j] = 0.f;
    lds_barrier();
    struct Ops {
        float q, k, u1;
        float4 sc;
    };
    const auto load_ops = [&](Ops &o, const RecBwdTile &T, const RecBwdTile &N, int tt, int nt) {
        o.q = T.qk[tt * 64 + half], o.k = T.qk[tt * 64 + 32 + half], o.sc = T.sc[tt], o.u1 = N.u[nt * 32 + pair];
    };
    const auto step = [&](const Ops &o, int tt, bool more, auto load) __attribute__((always_inline)) {
        const int p = tt & 1;
        lds_barrier();
        const float h = M.g[p][pair], P = M.P[p][pair];
        load();
        const float a = ready(-o.sc.x * fmaf(o.sc.y, h, P));
        rank1(G, h, o.q);
        rank1(G, a, o.k);
        if (more) M.Q[p ^ 1][32 + half] = sum_to_half(dot(G, o.u1));
    };
    for (int it = ntile - 1; it >= 0; it--) {
        const int nst = min(kTile, L - it * kTile);
        const RecBwdTile &T = M.tile[it & 1], &N = M.tile[it & 1 ^ 1];
        if (nst == kTile) {
            Ops ring[2];
            load_ops(ring[(kTile - 1) & 1], T, T, kTile - 1, kTile - 2);
#pragma unroll 1
            for (int tb = kTile - kUnroll; tb >= 0; tb -= kUnroll)
#pragma unroll
                for (int j = kUnroll - 1; j >= 0; j--)
                    step(ring[j & 1], tb + j, j || tb || it, [&] {
                        if (j > 1 || (j == 0 && tb)) load_ops(ring[(j + 1) & 1], T, T, tb + j - 1, tb + j - 2);
                        else if (j == 1) load_ops(ring[0], T, tb ? T : N, tb, tb ? tb - 1 : kTile - 1);
                    });
        } else {
#pragma unroll 1
            for (int tt = nst - 1; tt >= 0; tt--) {
                Ops o;
                load_ops(o, T, tt ? T : N, tt, tt ? tt - 1 : kTile - 1);
                step(o, tt, tt > 0 || it > 0, [] {});
            }
        }
    }
    lds_barrier();
}

// Loads, stores, the gradients of R.  In the steps of tile `it` (but the first): tile it + 1 is summed and stored, it - 1 goes to LDS, it - 2 is asked
// for, from the second step on: until the first step's barrier the others may still be at tile it + 1.
__device__ __forceinline__ void rec_bwd_y(RecBwdLds &M, const RecBwdArgs &g, int64_t seq, int lane) {
    constexpr int D = 32, NV4 = Geo<D>::NV4;
    const int n = (int)(seq / g.H), hd = (int)(seq % g.H), L = g.L, ntile = (L + kTile - 1) / kTile;
    const float *go = row(g.go, n, hd, 0);
    const int64_t first = seq * L * D;
    // Places are found again for each piece of work: kept for all of them in registers they would not fit.
    struct Place {
        int row, c4;
    };
    const auto place = [&] {
        int l = lane;
        asm volatile("" : "+v"(l));
        return Place{l / 8, l % 8 * 4};
    };
    rec_v4f pq[NV4], pk[NV4], pd[NV4], pg[NV4], py[NV4];
    float pb[NV4];
    const auto fetch = [&](int it) {
        const Place p = place();
#pragma unroll
        for (int i = 0; i < NV4; i++) {
            // rows beyond L hold the last one's values: they are no step's
            const int t = min(it * kTile + p.row + 8 * i, L - 1);
            const int64_t at = (int64_t)t * D + p.c4;
            pq[i] = *reinterpret_cast<const rec_v4f *>(g.q_act + first + at);
            pk[i] = *reinterpret_cast<const rec_v4f *>(g.k_act + first + at);
            pd[i] = *reinterpret_cast<const rec_v4f *>(g.vdiff + first + at);
            pg[i] = *reinterpret_cast<const rec_v4f *>(go + (int64_t)t * g.go.sL + p.c4);
            pb[i] = g.beta_act[seq * L + t];
            // row t of the delayed output is out[t-1], or the initial state for t = 0
            py[i] = *reinterpret_cast<const rec_v4f *>(t ? g.out + first + at - D : g.h_init + seq * D + p.c4);
        }
    };
    const auto commit_qk = [&](int it) {
        RecBwdTile &T = M.tile[it & 1];
        const Place p = place();
#pragma unroll
        for (int i = 0; i < NV4; i++) {
            const int tt = p.row + 8 * i;
            const rec_v4f x = pq[i], y = pk[i], xy = x * y;
            *reinterpret_cast<rec_v4f *>(T.qk + tt * 64 + p.c4) = x;
            *reinterpret_cast<rec_v4f *>(T.qk + tt * 64 + 32 + p.c4) = y;
            const float qk = row_reduce<D>((xy[0] + xy[1]) + (xy[2] + xy[3]), OpSum()), b = pb[i];
            if (p.c4 == 0) {
                T.sc[tt] = make_float4(b, qk, b * (1.f - b), 0.f);
                T.co[2 * tt] = 1.f, T.co[2 * tt + 1] = -b * qk;
            }
        }
    };
    const auto commit_v = [&](int it) {
        RecBwdTile &T = M.tile[it & 1];
#pragma unroll
        for (int i = 0; i < NV4; i++) {
            const int at = 4 * (lane + kWave * i);
            const rec_v4f d = pd[i];
            *reinterpret_cast<rec_v4f *>(T.go + at) = pg[i];
            *reinterpret_cast<rec_v4f *>(T.d + at) = d;
            *reinterpret_cast<rec_v4f *>(T.u + at) = pb[i] * d;
        }
    };
    const auto commit_y = [&](int it) {
        RecBwdTile &T = M.tile[it & 1];
#pragma unroll
        for (int i = 0; i < NV4; i++) {
            const int at = 4 * (lane + kWave * i);
            const rec_v4f x = py[i], h = {fast_tanh(x[0]), fast_tanh(x[1]), fast_tanh(x[2]), fast_tanh(x[3])};
            *reinterpret_cast<rec_v4f *>(M.y[it % 3] + at) = h;
            *reinterpret_cast<rec_v4f *>(T.dt + at) = 1.f - h * h;
        }
    };
    const auto flush = [&](int it, float *to, const float *from, int pitch) {
        const Place p = place();
#pragma unroll
        for (int i = 0; i < NV4; i++) {
            const int tt = p.row + 8 * i, t = it * kTile + tt;
            const rec_v4f x = *reinterpret_cast<const rec_v4f *>(from + tt * pitch + p.c4);
            if (t < L) *reinterpret_cast<rec_v4f *>(to + first + (int64_t)t * D + p.c4) = x;
        }
    };
    const auto store = [&](int it, int part) {
        const RecBwdTile &T = M.tile[it & 1];
        if (part == 0) flush(it, g.gqx, T.gqk, 64);
        else if (part == 1) flush(it, g.gkx, T.gqk + 32, 64);
        else {
            flush(it, g.gvx, T.gv, 32);
            const int t = it * kTile + lane;
            if (lane < kTile && t < L) g.gbx[seq * L + t] = T.gb[lane];
        }
    };
    // acc[x][m][n]: lane l, register r holds entry (16 m + 4 (l / 16) + r, 16 n + l % 16) of sum_t y_t (x) grad_x; accb the same
    // for y_t grad_bx in column 0
    rec_v4f acc[3][2][2], accb[2];
#pragma unroll
    for (int m = 0; m < 2; m++) {
        accb[m] = rec_v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int x = 0; x < 3; x++) acc[x][m][0] = acc[x][m][1] = rec_v4f{0.f, 0.f, 0.f, 0.f};
    }
    const auto sums = [&](int it, int j, int n) {      // of columns 16 n + l % 16, four steps to a matrix instruction: step 4 j + l / 16
        const RecBwdTile &T = M.tile[it & 1];
        int l = lane;
        asm volatile("" : "+v"(l));
        const int tt = 4 * j + l / 16, c = l % 16;
        const bool ok = it * kTile + tt < L;
        const float *const gqk = T.gqk + tt * 64 + 16 * n + c;
        const float x[3] = {ok ? gqk[0] : 0.f, ok ? gqk[32] : 0.f, ok ? T.gv[tt * 32 + 16 * n + c] : 0.f};
        const float xb = ok && c == 0 && n == 0 ? T.gb[tt] : 0.f;
#pragma unroll
        for (int m = 0; m < 2; m++) {
            const float y = ok ? M.y[it % 3][tt * D + 16 * m + c] : 0.f;
#pragma unroll
            for (int i = 0; i < 3; i++)
                if (n) acc[i][m][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(y, x[i], acc[i][m][1], 0, 0, 0);
                else acc[i][m][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(y, x[i], acc[i][m][0], 0, 0, 0);
            if (!n) accb[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(y, xb, accb[m], 0, 0, 0);
        }
    };
#pragma unroll 1
    for (int it = ntile - 1; it >= max(0, ntile - 2); it--) {
        fetch(it);
        commit_qk(it), commit_v(it), commit_y(it);
    }
    if (ntile > 2) fetch(ntile - 3);
    lds_barrier();
#pragma unroll 1
    for (int s = L - (ntile - 1) * kTile; s; s--) lds_barrier();      // the first tile's steps
#pragma unroll 1
    for (int it = ntile - 2; it >= 0; it--) {
        // a piece of work to a step; loads wait for the stores before them: as many steps between them as there are
        lds_barrier();
        if (it) commit_qk(it - 1);
        lds_barrier();
        if (it) commit_v(it - 1);
        lds_barrier();
        if (it) commit_y(it - 1);
        lds_barrier();
        if (it > 1) fetch(it - 2);
        lds_barrier();
#pragma unroll 1
        for (int j = 0; j < 3; j++) {
            store(it + 1, j);
            lds_barrier();
        }
#pragma unroll 1
        for (int j = 0; j < 4; j++) {
            sums(it + 1, j, 0);
            lds_barrier();
            sums(it + 1, j, 1);
            lds_barrier();
        }
    }
    lds_barrier();
#pragma unroll 1
    for (int j = 0; j < 4; j++) sums(0, j, 0), sums(0, j, 1);
#pragma unroll 1
    for (int j = 0; j < 3; j++) store(0, j);
    // this sequence's share of the parameter gradients: [gRq | gRk | gRv | grb], rows e, columns m
    float *ws = g.workspace + seq * (3 * D * D + D);
    const int r4 = lane / 16, c = lane % 16;
#pragma unroll
    for (int m = 0; m < 2; m++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int e = 16 * m + 4 * r4 + r;
#pragma unroll
            for (int x = 0; x < 3; x++)
#pragma unroll
                for (int k = 0; k < 2; k++) ws[x * D * D + e * D + 16 * k + c] = acc[x][m][k][r];
            if (c == 0) ws[3 * D * D + e] = accb[m][r];
        }
}

// NS sequences to a workgroup
template <int NS>
__global__ __launch_bounds__(kWave * 4 * NS) void k_rec_bwd_quad(RecBwdArgs g, int nseq) {
    extern __shared__ __align__(16) unsigned char quad_lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, role = wave / NS;
    const int64_t seq = (int64_t)blockIdx.x * NS + wave % NS;
    RecBwdLds &M = reinterpret_cast<RecBwdLds *>(quad_lds)[wave % NS];
    if (seq >= nseq) {      // spare waves only keep the barriers' count
        for (int t = g.L + 2; t; t--) lds_barrier();
        return;
    }
    if (role == 0) rec_bwd_x(M, g, seq, lane);
    else if (role == 1) rec_bwd_c(M, g, seq, lane);
    else if (role == 2) rec_bwd_d(M, g, seq, lane);
    else rec_bwd_y(M, g, seq, lane);
}

}  // namespace

bool reg_rec_supported(int D) { return D == 16 || D == 32; }

int reg_rec_fwd(fwp_view qx, fwp_view kx, fwp_view vx, fwp_view bx, const float *Rq,
                const float *Rk, const float *Rv, const float *rb, float *W, float *h, float *out,
                float *q_act, float *k_act, float *beta_act, float *vdiff, float *ckpt, int N,
                int H, int L, int D, int chunk, hipStream_t s) {
    const int nchunk = (L + chunk - 1) / chunk, nseq = N * H;
    auto launch = [&](auto kernel, int wpb) {
        hipLaunchKernelGGL(kernel, dim3((nseq + wpb - 1) / wpb), dim3(kWave * wpb), 0, s, qx, kx, vx, bx, Rq, Rk, Rv,
                           rb, W, h, out, q_act, k_act, beta_act, vdiff, ckpt, H, L, chunk, nchunk, nseq);
    };
    if (D == 16) launch(k_rec_fwd_reg<2, 1, 4>, 4);
    else {
        const RecFwdArgs g{qx, kx, vx, bx, Rq, Rk, Rv, rb, W, h, out, q_act, k_act, beta_act, vdiff, ckpt, H, L, chunk, nchunk, nseq};
        const auto go = [&](auto ns) {
            constexpr int NS = decltype(ns)::value;
            hipLaunchKernelGGL(k_rec_fwd_pair<NS>, dim3((nseq + NS - 1) / NS), dim3(2 * NS * kWave), 0, s, g);
        };
        // Two sequences to a workgroup while that is one workgroup on each CU, and from 1025 to 1536 sequences, three workgroups on a CU; else four (two-wave shares
        // of a CU are placed unevenly on its SIMDs once there is more than one).  20, 60 and 256 steps, workgroups of 2 / 4 / 8: 512 sequences
        // 13.0 / 13.5 / 19.6, 32.5 / 33.2 / 48.9 and 122 / 124 / 186 us, 1024 19.5 / 15.2 / 20.9, 47.8 / 34.8 / 49.6 and 181 / 131 / 191, 1536 20.5 / 21.1 / 21.6,
        // 49.4 / 50.1 / 50.8 and 187 / 193 / 197, 2048 23.9 / 23.4 / 24.6, 55.1 / 51.4 / 52.6 and 209 / 199 / 205.
        if (nseq <= 512 || (nseq > 1024 && nseq <= 1536)) go(std::integral_constant<int, 2>());
        else go(std::integral_constant<int, 4>());
    }
    return (int)hipGetLastError();
}

int reg_rec_bwd(const float *q_act, const float *k_act, const float *beta_act, const float *vdiff,
                const float *out, const float *h_init, fwp_view go, const float *Rq,
                const float *Rk, const float *Rv, const float *rb, const float *ckpt, float *gqx,
                float *gkx, float *gvx, float *gbx, float *workspace, int N, int H, int L, int D,
                int chunk, hipStream_t s) {
    const int nchunk = (L + chunk - 1) / chunk, nseq = N * H;
    auto launch = [&](auto kernel, int ns, size_t lds) {
        if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds))
            return (int)e;
        hipLaunchKernelGGL(kernel, dim3((nseq + ns - 1) / ns), dim3(kWave * 2 * ns), lds, s, q_act, k_act, beta_act,
                           vdiff, out, h_init, go, Rq, Rk, Rv, rb, ckpt, gqx, gkx, gvx, gbx, workspace, H, L, chunk,
                           nchunk, nseq);
        return (int)hipGetLastError();
    };
    // D = 32: the two-wave kernel has 1024 sequences on the chip at once, the four-wave one 512.  Where it needs half as many turns and the steps are few, what a turn
    // costs once weighs more than a step: two waves / four, 1024 sequences of 20, 60, 128, 160, 200 and 256 steps 36 / 39, 70 / 77, 132 / 136, 163 / 165, 204 / 201 and
    // 260 / 251 us; 2048 of 20, 128, 160 and 256 63 / 72, 265 / 269, 337 / 329 and 522 / 495; 771 of 20 and 200 34 / 39 and 197 / 198.
    if (D == 32 && L <= 160 && nseq > 768 && (nseq - 1) / 512 % 2 == 1) return launch(k_rec_bwd_pair<32, 4>, 4, 4 * sizeof(RecPairLds<32>));
    if (D == 32) {
        const RecBwdArgs g{q_act, k_act, beta_act, vdiff, out, h_init, go, Rq, Rk, Rv, rb, ckpt, gqx, gkx, gvx, gbx, workspace, H, L, chunk, nchunk};
        const auto run = [&](auto ns) {
            constexpr int NS = decltype(ns)::value;
            if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_rec_bwd_quad<NS>),
                                                   hipFuncAttributeMaxDynamicSharedMemorySize, (int)(NS * sizeof(RecBwdLds))))
                return (int)e;
            hipLaunchKernelGGL(k_rec_bwd_quad<NS>, dim3((nseq + NS - 1) / NS), dim3(4 * NS * kWave), NS * sizeof(RecBwdLds), s, g, nseq);
            return (int)hipGetLastError();
        };
        // Two sequences to a workgroup are 512 at a time; three (with spills) 768: 768 sequences of 20, 60 and 256 steps 31, 57 and 192 us where
        // workgroups of two take 39, 73 and 247, 1024 50, 102 and 370 and 39, 76 and 250.
        if (nseq > 512 && nseq <= 768) return run(std::integral_constant<int, 3>());
        return run(std::integral_constant<int, 2>());
    }
    // up to 512 sequences two to a workgroup (one workgroup on each CU), beyond that four
    if (nseq <= 512) return launch(k_rec_bwd_pair<16, 2>, 2, 2 * sizeof(RecPairLds<16>));
    return launch(k_rec_bwd_pair<16, 4>, 4, 4 * sizeof(RecPairLds<16>));
}

}  // namespace fwp
