// fp32 matrix products of the language model's layers on the bf16 matrix cores.
//
// An fp32 number is the sum of three bf16 numbers, x = h + m + l (h = bf16(x), m = bf16(x - h), l = the rest:
// 3 x 8 significant bits and their signs hold all 24), so a product of two fp32 numbers is the sum of nine bf16
// products.  Six of them are formed, h h', h m', m h', m m', h l', l h'; the three left out are below
// 2^-26 |x x'|, a quarter of the rounding of an fp32 product.  Sums are fp32, six roundings per 32 terms where a
// chain of fp32 multiply-adds has 32.  Measured against float64 (N(0,1) operands, 2-norm), with hipBLASLt's fp32 products of
// the same operands behind it: 32768 x 1024, K = 256 2.4e-7 (2.9e-7); 32768 x 256, K = 1024 4.9e-7 (5.7e-7); 32768 x 256,
// K = 32768 3.04e-6 (3.24e-6); 1024 x 256, K = 32768 in ranges 5.7e-7 (2.0e-6).
//
// bf16 has fp32's exponents: no scaling.  An operand that no bf16 number holds (infinity, NaN, the last 2^-9 below
// fp32's largest) leaves NaN or infinity in the sums: a tile with an element that is not finite is formed again on the fp32
// matrix instructions, which takes another one to one and a half times its time.  Parts of an operand below the
// smallest normal number count as zero: it is exact to 2^-24 of itself or to 2^-126, whichever is more.
//
// v_mfma_f32_16x16x32_bf16 makes 2.1 PFLOP/s with random operands (2.45 with zeros: the chip's power is the limit;
// the 32x32x16 form 1.8), i.e. 350 TFLOP/s of such fp32 products, where the fp32 matrix instructions make 155.
// The operands are split on their way from global memory to LDS, in the registers of the thread that loads
// them: 11 vector instructions per two numbers, 45 % of the matrix instructions' time in a 128 x 128 tile, and
// issued beside them by the other workgroups of the CU.  LDS holds 16-byte units of 8 consecutive k of one row,
// [plane][k / 8][row], so that a fragment is one ds_read_b128; an operand that is contiguous along its rows
// instead of along k is transposed in registers on the way.
//
// What bounds it: 32768 x 256, K = 1024 takes 89-93 us, 1.1 PFLOP/s of bf16 products.  Matrix instructions, fragment reads and
// barriers alone take 67 us (1.56 PFLOP/s), the LDS writes 15 us more, the split 5-10 us, loads that miss the cache 5 us; the
// clock falls to 1.8-1.9 GHz, so that cycles saved come back as time only in part.  Tried without gain: 256 x 128 tiles
// (256 registers, spills: 113 us), fragments fetched a dozen matrix instructions ahead (97 us), remainders by
// v_dot2_f32_bf16 (fewer instructions, 101 us, and it drops denormals).
#include "fwp_common.hpp"
#include "fwp_mfma.hpp"

namespace fwp {

typedef float v2f __attribute__((ext_vector_type(2)));
__device__ v2f llvm_raw_buffer_load_v2f32(v4i rsrc, int voffset, int soffset, int aux) __asm("llvm.amdgcn.raw.buffer.load.v2f32");

namespace {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

constexpr int kBK = 32;          // k per LDS tile
constexpr int kThreads = 256;
constexpr unsigned kOut = 0x80000000u;      // an offset beyond every buffer: reads as zero

__device__ __forceinline__ unsigned pack2(float a, float b) {
    const bf2 r = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(unsigned, r);
}
__device__ __forceinline__ float low_f(unsigned u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float high_f(unsigned u) { return __uint_as_float(u & 0xffff0000u); }

__device__ __forceinline__ v4i buffer_of(const float *base, int64_t floats) {
    const uint64_t a = reinterpret_cast<uint64_t>(base);
    return v4i{(int)(uint32_t)a, (int)(uint32_t)((a >> 32) & 0xffff), (int)(uint32_t)(floats * 4), 0x00020000};
}

__device__ __forceinline__ float lane_of(float x, int lane) {
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), lane));
}

template <int ROWS>
struct Planes {
    v4u u[3][kBK / 8][ROWS];
};

// The place of a row's unit in its k-chunk, such that no access meets a bank twice: a read takes lanes 0-3, 12-15, 20-23
// and 24-27 together (two chunks' rows: whole groups of four, whichever chunk), a write eight lanes, which hold two rows x
// four chunks (operands contiguous along k) or every other of sixteen rows (the others).  With rows in order and the
// chunks 32 bytes apart 420 of 1280 LDS cycles per tile step (x W^T), 770 of 1560 (g^T x) were conflicts; 32768 x 256,
// K = 1024: 4.7e7 -> 4.3e7 cycles of busy CUs, 95.0 -> 92.9 us.
__device__ __forceinline__ constexpr int unit_of(int row, int chunk) { return row ^ (2 * chunk) ^ ((row >> 3) & 1); }

// exp(x): 2^(x log2 e) by the hardware, x log2 e rounded to its nearest float and the rest of it as a factor: probabilities
// are off by at most 4 roundings, down to e^-70 (with x log2 e alone by 60 there; PyTorch's, through the logarithm, by 69).  Arguments below -150 give
// 0 as that one does (the rest of an infinity would be NaN); a NaN stays.
__device__ __forceinline__ float exp_of(float x) {
    constexpr float kLog2e = 1.44269504f, kLog2eRest = 1.92596299e-8f, kLn2 = 0.693147181f;
    x = x < -150.f ? -150.f : x;
    const float y = x * kLog2e, rest = fmaf(x, kLog2e, -y), e = __builtin_amdgcn_exp2f(y);
    return fmaf(e, fmaf(rest, kLn2, x * (kLog2eRest * kLn2)), e);
}

// What turns stored logits into the gradient of the loss as an operand is loaded:
// (exp(logit - shift) * scale - [vocabulary entry == target]) * gloss of the token, 0 for an ignored target, NaN for one that
// is no word.
// shift and scale: the largest logit and 1 / the sum of exp(logit - largest) (`stats`, exact where a token's probability
// is near 1 and its logit large), or the log-sum-exp and 1 (`lse`).
struct NllArgs {
    const float *lse, *stats, *gloss;
    const int64_t *target;
    int vocab;
};

constexpr int64_t kIgnored = -100;      // torch.nn.functional.cross_entropy's ignore_index

struct NllToken {
    float shift, scaled, g;      // scaled: scale * gloss
    int hit;
};

__device__ __forceinline__ NllToken nll_token(const NllArgs &a, int token) {
    NllToken t;
    const int64_t want = a.target[token];
    t.hit = (int)want;
    t.g = want == kIgnored ? 0.f : want >= 0 && want < a.vocab ? a.gloss[token] : NAN;
    const float2 s = a.stats ? reinterpret_cast<const float2 *>(a.stats)[token] : make_float2(a.lse[token], 1.f);
    t.shift = s.x;
    t.scaled = s.y * t.g;
    return t;
}

__device__ __forceinline__ float nll_grad(float logit, float shift, float scaled, float g, bool hit) {
    return fmaf(exp_of(logit - shift), scaled, hit ? -g : 0.f);
}

// One operand's share of the loads and LDS writes of a thread.  KC: rows are contiguous along k; a task is 8
// consecutive k of one row (two 16-byte loads, one unit per plane).  Otherwise contiguous along the rows; a
// task is VEC consecutive rows x 8 k (8 loads, VEC units per plane).
// NLL: the operand is the loss gradient, formed from the logits; tokens are the rows (KC) or k.
template <bool KC, int ROWS, bool NLL>
struct Operand {
    static constexpr int kChunks = kBK / 8;
    static constexpr int VEC = KC ? 1 : ROWS * kChunks / kThreads;          // 2 at 128 rows, 1 at 64
    static constexpr int kTasks = KC ? ROWS * kChunks / kThreads : 1;
    static_assert(KC ? kTasks >= 1 : (VEC == 1 || VEC == 2), "a whole number of tasks per thread");
    float x[kTasks][8 * VEC];
    unsigned off[kTasks];
    // the tokens' values for the loss gradient: of this task's row (KC), or of the wave's k-chunk, token j in
    // the lanes with lane % 8 == j
    NllToken token[NLL ? kTasks : 1];

    static __device__ __forceinline__ int row_of(int t) { return KC ? t / kChunks : (t % (ROWS / VEC)) * VEC; }
    static __device__ __forceinline__ int chunk_of(int t) { return KC ? t % kChunks : t / (ROWS / VEC); }

    __device__ __forceinline__ void init(int tid, int64_t ld, int row0, int rows, const NllArgs &nll) {
#pragma unroll
        for (int i = 0; i < kTasks; i++) {
            const int r = row_of(tid + i * kThreads), c = chunk_of(tid + i * kThreads);
            off[i] = (unsigned)(KC ? r * ld + 8 * c : 8 * c * ld + r) * 4;
            if constexpr (NLL && KC) token[i] = nll_token(nll, min(row0 + r, rows - 1));
        }
    }
    // P: the tile's first row at k = 0, `left` rows from there, k0 .. min(k0 + kBK, K)
    __device__ __forceinline__ void load(const float *P, int64_t ld, int left, int tid, int k0, int K, const NllArgs &nll) {
        if constexpr (KC) {
            const v4i rs = buffer_of(P + k0, (int64_t)(min(left, ROWS) - 1) * ld + (K - k0));
#pragma unroll
            for (int i = 0; i < kTasks; i++) {
                const int k = k0 + 8 * chunk_of(tid + i * kThreads);
                const v4f a = llvm_raw_buffer_load_v4f32(rs, (int)(k < K ? off[i] : kOut), 0, 0),
                          b = llvm_raw_buffer_load_v4f32(rs, (int)(k + 4 < K ? off[i] + 16 : kOut), 0, 0);
#pragma unroll
                for (int j = 0; j < 4; j++) x[i][j] = a[j], x[i][4 + j] = b[j];
            }
        } else {
            if constexpr (NLL) token[0] = nll_token(nll, min(k0 + 8 * chunk_of(tid) + tid % 8, K - 1));
            const v4i rs = buffer_of(P + (int64_t)k0 * ld, (int64_t)(min(K - k0, kBK) - 1) * ld + left);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                if constexpr (VEC == 1) {
                    x[0][j] = llvm_raw_buffer_load_f32(rs, (int)off[0], (int)(j * ld * 4), 0);
                } else {
                    const v2f a = llvm_raw_buffer_load_v2f32(rs, (int)off[0], (int)(j * ld * 4), 0);
                    x[0][j] = a[0], x[0][8 + j] = a[1];
                }
            }
        }
    }
    // What load() brought: zeros beyond K (a row contiguous along k runs on into the next row there), and the
    // loss gradient in place of the logits
    __device__ __forceinline__ void finish(int tid, int row0, int k0, int K, const NllArgs &nll) {
        if constexpr (KC) {
            const bool tail = k0 + kBK > K;
#pragma unroll
            for (int i = 0; i < kTasks; i++) {
                const int k = k0 + 8 * chunk_of(tid + i * kThreads);
                if constexpr (NLL)
#pragma unroll
                    for (int j = 0; j < 8; j++)
                        x[i][j] = nll_grad(x[i][j], token[i].shift, token[i].scaled, token[i].g, token[i].hit == k + j);
                if (tail)
#pragma unroll
                    for (int j = 0; j < 8; j++) x[i][j] = k + j < K ? x[i][j] : 0.f;
            }
        } else if constexpr (NLL) {
            static_assert(ROWS / VEC == 64, "a k-chunk per wave");
            const int k = k0 + 8 * chunk_of(tid), r = row0 + row_of(tid);
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const float shift = lane_of(token[0].shift, j), scaled = lane_of(token[0].scaled, j), g = lane_of(token[0].g, j);
                const int h = __builtin_amdgcn_readlane(token[0].hit, j);
#pragma unroll
                for (int c = 0; c < VEC; c++) {
                    // a token beyond K has the last one's values beside a logit of 0: its exponential may be infinite
                    const float d = nll_grad(x[0][8 * c + j], shift, scaled, g, h == r + c);
                    x[0][8 * c + j] = k + j < K ? d : 0.f;
                }
            }
        }
    }
    __device__ __forceinline__ void store(Planes<ROWS> &L, int tid) const {
#pragma unroll
        for (int i = 0; i < kTasks; i++)
#pragma unroll
            for (int c = 0; c < VEC; c++) {
                v4u h, m, l;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float a = x[i][8 * c + 2 * j], b = x[i][8 * c + 2 * j + 1];
                    h[j] = pack2(a, b);
                    const float ra = a - low_f(h[j]), rb = b - high_f(h[j]);
                    m[j] = pack2(ra, rb);
                    l[j] = pack2(ra - low_f(m[j]), rb - high_f(m[j]));
                }
                const int r = row_of(tid + i * kThreads) + c, ch = chunk_of(tid + i * kThreads);
                const int at = unit_of(r, ch);
                L.u[0][ch][at] = h;
                L.u[1][ch][at] = m;
                L.u[2][ch][at] = l;
            }
    }
    // fp32 as it is: 16-byte units of 4 consecutive k of one row, [k / 4][row], in the same memory
    static __device__ __forceinline__ v4f *plain(Planes<ROWS> &L) { return reinterpret_cast<v4f *>(&L); }
    __device__ __forceinline__ void store_plain(Planes<ROWS> &L, int tid) const {
#pragma unroll
        for (int i = 0; i < kTasks; i++)
#pragma unroll
            for (int c = 0; c < VEC; c++)
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const float *const y = x[i] + 8 * c + 4 * j;
                    plain(L)[(2 * chunk_of(tid + i * kThreads) + j) * ROWS + row_of(tid + i * kThreads) + c] = v4f{y[0], y[1], y[2], y[3]};
                }
    }
};

struct GemmArgs {
    const float *A, *B;
    float *C;                    // the result, or (several k ranges) one M x N partial result per range, `part` floats apart
    int64_t lda, ldb, ldc, part;
    int M, N, K;
    int ks;                      // k per range (a multiple of kBK)
    int vec;                     // C, residual and gate can be accessed 16 bytes at a time
    int tm, tn;                  // tiles
    float *colsum;               // sums over k of A's rows, per range [M] (A contiguous along its rows), or NULL
    fwp_mm_epilogue epi;         // applied here when there is one range
    NllArgs nll;
    // per tile of columns and row: the largest logit and the sum of exp(logit - largest); logits of the targets
    float *part_max, *part_sum, *hit;
};

enum { kPlain = 0, kLse = 1, kGrad = 2 };

// everything but the bias
__device__ __forceinline__ float apply(const fwp_mm_epilogue &e, float x, int64_t at) {
    if (e.relu) x = relu(x);
    if (e.residual) x += e.residual[at];
    if (e.gate) x = gated(e.gate[at], x);
    return x;
}

template <int X>
__device__ __forceinline__ float rotated(float x) {      // within the 16 lanes of a DPP row
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(x), 0x120 + X, 0xf, 0xf, true));
}

// LDS accesses of one wave execute in order; this keeps the compiler from moving them across.
__device__ __forceinline__ void wave_lds_order() { asm volatile("" ::: "memory"); }

// What a sum of exp(logit - m) is multiplied with to become one of exp(logit - big).  A part of the vocabulary with no
// logit but -infinity (masked words; columns beyond the last) has m = -infinity and the sum 0, or NaN if there
// was one: it stays as it is (exp(-infinity + infinity) would make it NaN).
__device__ __forceinline__ float to_max(float m, float big) { return m == -INFINITY ? 1.f : exp_of(m - big); }

// The largest of a row's logits and the sum of exp(logit - largest): four logits per lane, LANES (8 or 16) lanes per row.
template <int LANES>
__device__ __forceinline__ void lse_of_row(float4 v, int n, int N, int lane, float *out, int at, int pitch) {
    if (n + 3 >= N) {
        v.x = n < N ? v.x : -INFINITY, v.y = n + 1 < N ? v.y : -INFINITY;
        v.z = n + 2 < N ? v.z : -INFINITY, v.w = -INFINITY;
    }
    float m = fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w));
    if constexpr (LANES == 16) {
        m = fmaxf(m, rotated<8>(m));
        m = fmaxf(m, rotated<4>(m)), m = fmaxf(m, rotated<2>(m)), m = fmaxf(m, rotated<1>(m));
    } else {
#pragma unroll
        for (int o = 4; o >= 1; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
    }
    const float z = m == -INFINITY ? 0.f : m;
    float s = (exp_of(v.x - z) + exp_of(v.y - z)) + (exp_of(v.z - z) + exp_of(v.w - z));
    if constexpr (LANES == 16) {
        s += rotated<8>(s);
        s += rotated<4>(s), s += rotated<2>(s), s += rotated<1>(s);
    } else {
#pragma unroll
        for (int o = 4; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    }
    if (lane % LANES == 0) out[at] = m, out[at + pitch] = s;
}

// Three waves per SIMD, three workgroups on a CU: the products with the loss's gradient are held to 168 registers for it
// (174 without the bound; one is spilled, outside the loop).
//
// BM x BN tile of four waves (two by two), each wave (BM/2) x (BN/2) in 16 x 16 MFMA tiles.
template <bool AKC, bool BKC, int BM, int BN, int MODE>
__global__ __launch_bounds__(kThreads, 3) void k_gemm(GemmArgs g) {
    constexpr int WM = BM / 2, WN = BN / 2, MT = WM / 16, NT = WN / 16;
    __shared__ Planes<BM> La;
    __shared__ Planes<BN> Lb;
    __shared__ int odd_waves[4];
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int wm = (wave % 2) * WM, wn = (wave / 2) * WN;
    // workgroups go round the 8 XCDs: each XCD gets a run of neighbouring tiles (a row of tiles reads the same
    // rows of A, through that XCD's L2)
    const int total = g.tm * g.tn, xcd = blockIdx.x % 8, each = total / 8, rest = total % 8;
    const int id = xcd * each + min(xcd, rest) + blockIdx.x / 8;
    const int m0 = (id / g.tn) * BM, n0 = (id % g.tn) * BN;
    const int kb = blockIdx.y * g.ks, ke = min(g.K, kb + g.ks);
    Operand<AKC, BM, MODE == kGrad> a;
    Operand<BKC, BN, false> b;
    a.init(tid, g.lda, m0, g.M, g.nll);
    b.init(tid, g.ldb, n0, g.N, g.nll);
    const float *Ap = AKC ? g.A + (int64_t)m0 * g.lda : g.A + m0;
    const float *Bp = BKC ? g.B + (int64_t)n0 * g.ldb : g.B + n0;
    const int ml = g.M - m0, nl = g.N - n0;
    constexpr int CV = AKC ? 1 : Operand<AKC, BM, MODE == kGrad>::VEC;
    float csum[CV];
#pragma unroll
    for (int c = 0; c < CV; c++) csum[c] = 0.f;
    const bool sums = !AKC && g.colsum && n0 == 0;
    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    const int lr = lane % 16, lc = lane / 16, lu = unit_of(lr, lc);
    a.load(Ap, g.lda, ml, tid, kb, ke, g.nll);
    b.load(Bp, g.ldb, nl, tid, kb, ke, g.nll);
    for (int k0 = kb; k0 < ke; k0 += kBK) {
        a.finish(tid, m0, k0, ke, g.nll);
        b.finish(tid, n0, k0, ke, g.nll);
        if constexpr (!AKC) {
            if (sums)
#pragma unroll
                for (int c = 0; c < CV; c++)
#pragma unroll
                    for (int j = 0; j < 8; j++) csum[c] += a.x[0][8 * c + j];
        }
        a.store(La, tid);
        b.store(Lb, tid);
        lds_barrier();
        if (k0 + kBK < ke) {
            a.load(Ap, g.lda, ml, tid, k0 + kBK, ke, g.nll);
            b.load(Bp, g.ldb, nl, tid, k0 + kBK, ke, g.nll);
        }
        // the products in an order in which three fragment sets are live at a time (six in the order of their size:
        // 178 registers instead of 162, two workgroups on a CU instead of three)
        bf8 a1[MT], a2[MT], b1[NT], b2[NT];
        const auto read_a = [&](bf8 *d, int p) {
#pragma unroll
            for (int i = 0; i < MT; i++) d[i] = __builtin_bit_cast(bf8, La.u[p][lc][wm + 16 * i + lu]);
        };
        const auto read_b = [&](bf8 *d, int p) {
#pragma unroll
            for (int j = 0; j < NT; j++) d[j] = __builtin_bit_cast(bf8, Lb.u[p][lc][wn + 16 * j + lu]);
        };
        const auto products = [&](const bf8 *x, const bf8 *y) {
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x[i], y[j], acc[i][j], 0, 0, 0);
        };
        read_a(a1, 2), read_b(b1, 0), products(a1, b1);      // l h'
        read_a(a2, 1), products(a2, b1);                     // m h'
        read_b(b2, 1), products(a2, b2);                     // m m'
        read_a(a1, 0), products(a1, b2);                     // h m'
        products(a1, b1);                                    // h h'
        read_b(b2, 2), products(a1, b2);                     // h l'
        lds_barrier();
    }

    // An element that is not finite (0 times it is NaN): the tile once more from the fp32 operands
    float odd = 0.f;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) odd = fmaf(acc[i][j][r], 0.f, odd);
    const bool wave_odd = __any(odd != 0.f);
    if (lane == 0) odd_waves[wave] = wave_odd;
    __syncthreads();
    if (odd_waves[0] | odd_waves[1] | odd_waves[2] | odd_waves[3]) {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        for (int k0 = kb; k0 < ke; k0 += kBK) {
            a.load(Ap, g.lda, ml, tid, k0, ke, g.nll);
            b.load(Bp, g.ldb, nl, tid, k0, ke, g.nll);
            a.finish(tid, m0, k0, ke, g.nll);
            b.finish(tid, n0, k0, ke, g.nll);
            a.store_plain(La, tid);
            b.store_plain(Lb, tid);
            __syncthreads();
            // lane (lc, lr) holds four consecutive k of row lr; register r of both operands is an instruction's four k
#pragma unroll 1
            for (int s = 0; s < kBK / 4; s += 4) {
                v4f y[NT];
#pragma unroll
                for (int j = 0; j < NT; j++) y[j] = b.plain(Lb)[(s + lc) * BN + wn + 16 * j + lr];
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const v4f x = a.plain(La)[(s + lc) * BM + wm + 16 * i + lr];
#pragma unroll
                    for (int r = 0; r < 4; r++)
#pragma unroll
                        for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[r], y[j][r], acc[i][j], 0, 0, 0);
                }
            }
            __syncthreads();
        }
    }

    // acc[i][j][r] = C[m0 + wm + 16 i + 4 lc + r][n0 + wn + 16 j + lr]
    if constexpr (!AKC) {
        if (sums) {      // the threads of a row pair's four k-chunks
            float *s = reinterpret_cast<float *>(&La);
            using Op = Operand<AKC, BM, MODE == kGrad>;
#pragma unroll
            for (int c = 0; c < CV; c++) s[Op::chunk_of(tid) * BM + Op::row_of(tid) + c] = csum[c];
            __syncthreads();
            for (int r = tid; r < min(BM, ml); r += kThreads)
                g.colsum[(int64_t)blockIdx.y * g.M + m0 + r] = (s[r] + s[BM + r]) + (s[2 * BM + r] + s[3 * BM + r]);
        }
    }
    // A wave turns its rows round through LDS (its own: no barrier), 16 at a time, so that they leave, and the
    // residual and the gate arrive, 16 bytes per lane: 4-byte accesses in the MFMA layout, 64-byte pieces of rows, cost
    // 112 us where this costs 90 at 32768 x 1024, K = 256.
    constexpr int kPitch = WN + 4;
    static_assert(4 * 16 * kPitch <= (int)(sizeof(La) / 4), "four waves' strips fit the first operand's planes");
    float *const strip = reinterpret_cast<float *>(&La) + wave * 16 * kPitch;
    constexpr int kLanes = WN / 4, kRows = 64 / kLanes;      // lanes per row, rows per access
    const int c4 = (lane % kLanes) * 4, n = n0 + wn + c4;
    const bool vec = g.vec && n + 3 < g.N;
    if constexpr (!AKC) __syncthreads();      // the column sums' reads of the same memory
    float bias[4];
#pragma unroll
    for (int e = 0; e < 4; e++) bias[e] = g.epi.bias && n + e < g.N && (gridDim.y == 1) ? g.epi.bias[n + e] : 0.f;
    float *const C = g.C + blockIdx.y * g.part;
    const bool one = gridDim.y == 1;
    float *const sums_of = reinterpret_cast<float *>(&Lb);       // kLse: [2][column half][row]
#pragma unroll
    for (int i = 0; i < MT; i++) {
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) strip[(4 * lc + r) * kPitch + 16 * j + lr] = acc[i][j][r];
        wave_lds_order();
#pragma unroll
        for (int q = 0; q < 16 / kRows; q++) {
            const int row = kRows * q + lane / kLanes, m = m0 + wm + 16 * i + row;
            float4 v = *reinterpret_cast<const float4 *>(strip + row * kPitch + c4);
            v.x += bias[0], v.y += bias[1], v.z += bias[2], v.w += bias[3];
            if constexpr (MODE == kLse) {
                lse_of_row<kLanes>(v, n, g.N, lane, sums_of, (wave / 2) * BM + wm + 16 * i + row, 2 * BM);
                if (g.hit && m < g.M) {
                    const int at = (int)g.nll.target[m] - n;
                    if (at >= 0 && at < 4 && n + at < g.N) g.hit[m] = at == 0 ? v.x : at == 1 ? v.y : at == 2 ? v.z : v.w;
                }
                if (!g.C) continue;
            }
            if (m >= g.M) continue;
            const int64_t at = (int64_t)m * g.ldc + n;
            if (vec) {
                if (one) {
                    if (g.epi.relu) v = make_float4(relu(v.x), relu(v.y), relu(v.z), relu(v.w));
                    if (g.epi.residual) {
                        const float4 y = *reinterpret_cast<const float4 *>(g.epi.residual + at);
                        v.x += y.x, v.y += y.y, v.z += y.z, v.w += y.w;
                    }
                    if (g.epi.gate) {
                        const float4 y = *reinterpret_cast<const float4 *>(g.epi.gate + at);
                        v = make_float4(gated(y.x, v.x), gated(y.y, v.y), gated(y.z, v.z), gated(y.w, v.w));
                    }
                }
                *reinterpret_cast<float4 *>(C + at) = v;
            } else {
                const float w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < g.N) C[at + e] = one ? apply(g.epi, w[e], at + e) : w[e];
            }
        }
        wave_lds_order();
    }
    if constexpr (MODE == kLse) {
        __syncthreads();
        for (int row = tid; row < min(BM, ml); row += kThreads) {
            const float m1 = sums_of[row], m2 = sums_of[BM + row], mx = fmaxf(m1, m2);
            const int64_t at = (int64_t)(id % g.tn) * g.M + m0 + row;
            g.part_max[at] = mx;
            g.part_sum[at] = sums_of[2 * BM + row] * to_max(m1, mx) + sums_of[3 * BM + row] * to_max(m2, mx);
        }
    }
}

// C[M,N] = the sum of `ranges` partial results `stride` floats apart (whole 16-byte groups: the last may reach beyond M N),
// with the epilogue; four threads share four neighbouring elements, a quarter of the ranges each, and add up in a
// fixed order.  The workgroups behind them do the same for the column sums of A ([ranges][M] behind the partial results).
__global__ __launch_bounds__(kThreads) void k_gemm_reduce(const float *__restrict__ part, float *__restrict__ C,
                                                          int64_t total, int64_t stride, int M, int N, int ranges,
                                                          fwp_mm_epilogue epi) {
    __shared__ float4 s[4][64];
    const int e = threadIdx.x % 64, q = threadIdx.x / 64;
    const int64_t blocks = (stride / 4 + 63) / 64;
    if (blockIdx.x >= blocks) {
        const float *const col = part + ranges * stride;
        const int m = (int)(blockIdx.x - blocks) * 64 + e;
        float x = 0.f;
        if (m < M) {
#pragma unroll 4
            for (int r = q; r < ranges; r += 4) x += col[(int64_t)r * M + m];
        }
        s[q][e].x = x;
        __syncthreads();
        if (q == 0 && m < M) epi.colsum[m] = (s[0][e].x + s[1][e].x) + (s[2][e].x + s[3][e].x);
        return;
    }
    const int64_t at = ((int64_t)blockIdx.x * 64 + e) * 4;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (at < total) {
#pragma unroll 4
        for (int r = q; r < ranges; r += 4) {
            const float4 y = *reinterpret_cast<const float4 *>(part + r * stride + at);
            x.x += y.x, x.y += y.y, x.z += y.z, x.w += y.w;
        }
    }
    s[q][e] = x;
    __syncthreads();
    if (q || at >= total) return;
    for (int o = 1; o < 4; o++) {
        const float4 y = s[o][e];
        x.x += y.x, x.y += y.y, x.z += y.z, x.w += y.w;
    }
    float v[4] = {x.x, x.y, x.z, x.w};
    const int n = (int)(at % N);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (at + i >= total) break;
        if (epi.bias) v[i] += epi.bias[N % 4 ? (int)((at + i) % N) : n + i];
        v[i] = apply(epi, v[i], at + i);
    }
    if (at + 3 < total) *reinterpret_cast<float4 *>(C + at) = make_float4(v[0], v[1], v[2], v[3]);
    else
        for (int i = 0; at + i < total; i++) C[at + i] = v[i];
}

struct Plan {
    bool wide;           // 128 x 128 tiles, else 64 x 64
    int tm, tn, ranges, ks;
};

// 128 x 128 tiles where they fill the chip (two workgroups on each of 256 CUs) or where k can be cut into ranges
// until they do; the partial results of a range cost a pass over M x N each way, so a range is no shorter than 256 of k.
// Without ranges to cut, fewer tiles than CUs: 64 x 64.
Plan plan_of(int M, int N, int K, bool may_cut) {
    Plan p;
    const auto tiles = [&](int b) { return (int64_t)((M + b - 1) / b) * ((N + b - 1) / b); };
    p.wide = tiles(128) >= 256 || (may_cut && tiles(128) * (K / 256) >= 256);
    const int b = p.wide ? 128 : 64;
    p.tm = (M + b - 1) / b;
    p.tn = (N + b - 1) / b;
    int64_t ranges = 1;
    if (may_cut) {
        ranges = 512 / (tiles(b));
        if (ranges > K / 256) ranges = K / 256;
        if (ranges < 1) ranges = 1;
    }
    p.ks = (int)((K + ranges - 1) / ranges + kBK - 1) / kBK * kBK;
    p.ranges = (K + p.ks - 1) / p.ks;
    return p;
}

template <bool AKC, bool BKC, int MODE>
void launch(const GemmArgs &g, const Plan &p, hipStream_t s) {
    const dim3 grid((unsigned)(p.tm * p.tn), (unsigned)p.ranges);
    if (p.wide) hipLaunchKernelGGL((k_gemm<AKC, BKC, 128, 128, MODE>), grid, dim3(kThreads), 0, s, g);
    else hipLaunchKernelGGL((k_gemm<AKC, BKC, 64, 64, MODE>), grid, dim3(kThreads), 0, s, g);
}

bool aligned(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// a partial result, in whole 16-byte groups
int64_t part_of(int M, int N) { return ((int64_t)M * N + 3) / 4 * 4; }

}  // namespace

int64_t matmul_workspace(int M, int N, int K) {
    const Plan p = plan_of(M, N, K, true);
    return p.ranges > 1 ? p.ranges * (part_of(M, N) + M) : 0;
}

int matmul(int layout, const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int64_t ldc, int M, int N,
           int K, const fwp_mm_epilogue &epi, float *workspace, const NllView *nll, hipStream_t s) {
    GemmArgs g{};
    g.A = A, g.B = B, g.lda = lda, g.ldb = ldb, g.M = M, g.N = N, g.K = K, g.epi = epi;
    if (nll) g.nll = NllArgs{nll->lse, nll->stats, nll->gloss, nll->target, nll->vocab};
    const Plan p = plan_of(M, N, K, workspace && ldc == N && aligned(C) && aligned(workspace));
    g.ks = p.ks, g.tm = p.tm, g.tn = p.tn;
    const bool cut = p.ranges > 1;
    g.C = cut ? workspace : C;
    g.ldc = cut ? N : ldc;
    g.part = part_of(M, N);
    g.vec = g.ldc % 4 == 0 && aligned(g.C) && aligned(epi.residual) && aligned(epi.gate);
    float *const col = cut ? workspace + p.ranges * g.part : epi.colsum;
    g.colsum = layout == FWP_MM_TN && epi.colsum ? col : nullptr;
    if (layout == FWP_MM_NT) launch<true, true, kPlain>(g, p, s);
    else if (layout == FWP_MM_NN && !nll) launch<true, false, kPlain>(g, p, s);
    else if (layout == FWP_MM_NN) launch<true, false, kGrad>(g, p, s);
    else if (!nll) launch<false, false, kPlain>(g, p, s);
    else launch<false, false, kGrad>(g, p, s);
    if (cut) {
        const int64_t total = (int64_t)M * N, blocks = (g.part / 4 + 63) / 64 + (g.colsum ? (M + 63) / 64 : 0);
        hipLaunchKernelGGL(k_gemm_reduce, dim3((unsigned)blocks), dim3(kThreads), 0, s, workspace, C, total, g.part, M, N, p.ranges, epi);
    }
    return (int)hipGetLastError();
}

namespace {

// loss = (largest logit - logit of the target) + log(sum of exp(logit - largest)) (0 for an ignored target, NaN for one
// that is no word), from the tiles' maxima and sums; four threads share a row, a quarter of the tiles each.  The difference comes first: added to
// the logarithm first, a large logit would round it off (a loss of 1e-3 at a logit of 20 by half a percent).
__global__ __launch_bounds__(kThreads) void k_nll(const float *__restrict__ part_max, const float *__restrict__ part_sum,
                                                  const float *__restrict__ hit, const float *__restrict__ logits,
                                                  const int64_t *__restrict__ target, float *__restrict__ loss, float *__restrict__ lse,
                                                  float *__restrict__ stats, int rows, int vocab, int tiles) {
    __shared__ float sm[4][64], ss[4][64];
    const int e = threadIdx.x % 64, q = threadIdx.x / 64, m = blockIdx.x * 64 + e;
    float mx = -INFINITY, s = 0.f;
    if (m < rows)
        for (int t = q; t < tiles; t += 4) {
            const float x = part_max[(int64_t)t * rows + m], y = part_sum[(int64_t)t * rows + m], big = fmaxf(mx, x);
            s = s * to_max(mx, big) + y * to_max(x, big);
            mx = big;
        }
    sm[q][e] = mx;
    ss[q][e] = s;
    __syncthreads();
    if (q || m >= rows) return;
    for (int o = 1; o < 4; o++) {
        const float x = sm[o][e], big = fmaxf(mx, x);
        s = s * to_max(mx, big) + ss[o][e] * to_max(x, big);
        mx = big;
    }
    const float l = logf(s);
    const int64_t want = target[m];
    if (lse) lse[m] = mx + l;
    if (stats) *reinterpret_cast<float2 *>(stats + 2 * (int64_t)m) = make_float2(mx, 1.f / s);
    // a row of -infinities alone: NaN
    loss[m] = want == kIgnored ? 0.f : want >= 0 && want < vocab ? (mx - (logits ? logits[(int64_t)m * vocab + want] : hit[m])) + l : NAN;
}

}  // namespace

int64_t nll_workspace(int rows, int vocab) { return (int64_t)((vocab + 63) / 64) * rows * 2 + rows; }

int nll_fwd(const float *x, const float *W, const float *bias, const int64_t *target, float *logits, float *loss,
            float *lse, float *stats, float *workspace, int rows, int vocab, int dim, hipStream_t s) {
    GemmArgs g{};
    g.A = x, g.B = W, g.lda = dim, g.ldb = dim, g.M = rows, g.N = vocab, g.K = dim, g.C = logits, g.ldc = vocab;
    g.epi.bias = bias;
    g.nll.target = target;
    const Plan p = plan_of(rows, vocab, dim, false);
    g.ks = p.ks, g.tm = p.tm, g.tn = p.tn;
    g.part_max = workspace;
    g.part_sum = workspace + (int64_t)p.tn * rows;
    g.hit = logits ? nullptr : g.part_sum + (int64_t)p.tn * rows;
    g.vec = vocab % 4 == 0 && aligned(logits);
    launch<true, true, kLse>(g, p, s);
    hipLaunchKernelGGL(k_nll, dim3((rows + 63) / 64), dim3(kThreads), 0, s, g.part_max, g.part_sum, g.hit, logits, target, loss,
                       lse, stats, rows, vocab, p.tn);
    return (int)hipGetLastError();
}

}  // namespace fwp
