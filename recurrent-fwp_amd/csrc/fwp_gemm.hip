// fp32 matrix products of the language model's layers on the 16-bit matrix cores, each operand split into a few 16-bit
// numbers, their products summed in fp32.
//
// Half2 (K >= 128): x s = h + m, h = fp16(x s), m = fp16(x s - h), three products m h', h m', h h'.  s is a power of two for each row
// of an operand (the rows of C, the columns of C).  h and m hold x to 2^-23 of itself; m m' is below
// 2^-22 |x x'|.  That is 7e-8 of a product, at random, where a sum's roundings, three per 32 terms, make more: relative error
// against float64 (N(0,1) operands, 2-norm; in brackets Bf16x3, then hipBLASLt's fp32): K = 128 1.39e-7 (1.61e-7), 32768 x 1024, K = 256
// 1.87e-7 (2.36e-7, 2.9e-7); 32768 x 256, K = 1024 3.6e-7 (4.9e-7, 5.7e-7); 1024 x 256, K = 32768 in ranges 3.9e-7 (5.75e-7, 2.0e-6).
// fp16 has few exponents: s brings a row's largest element so far to [2^13, 2^14).  One beyond 65504 / s (a row that grows fourfold
// or more along k) moves s, and the row's results so far with it.  An element below about 2^-20 of its row's largest would lose bits: the
// waves look for those, and what two numbers leave of them is multiplied apart, so that an element counts to 2^-19 of itself or better
// whatever is in its row (a result may be made of small elements alone).  The search costs 7 us of 71, 32768 x 256, K = 1024.
// Where small elements are many (tokens' gradients, features of very different sizes) that is left: step by step kernels go on with Bf16x3,
// those with B's rows kept make the products of the small elements once more, small products are formed again on fp32.  x^T y, 1024 x 256, K = 32768,
// the size of k exp(a N(0,1)), a = 0 / 1.5 / 3 / 5: 80 / 102 / 103 / 98 us (Bf16x3 alone 96; element by element 84 / 122 / 301 / 460).
//
// Bf16x3 (smaller K, and the loss's gradient): x = h + m + l (h = bf16(x), m = bf16(x - h), l = the rest: 3 x 8 significant bits and
// their signs hold all 24), six products, h h', h m', m h', m m', h l', l h'; the three left out are below 2^-26 |x x'|.  bf16
// has fp32's exponents: no scaling.  Parts of an operand below the smallest normal number count as zero: it is exact to
// 2^-24 of itself or to 2^-126, whichever is more.
//
// An operand that the 16-bit numbers cannot hold (infinity, NaN, for bf16 the last 2^-9 below fp32's largest) leaves NaN or infinity in
// the sums: a tile with an element that is not finite is formed again on the fp32 matrix instructions, a third of the rate or less.
//
// v_mfma_f32_16x16x32_bf16 makes 1.7-2.1 PFLOP/s with random operands and the f16 form 1.5 (2.45 with zeros: the chip's power is
// the limit), i.e. 490 TFLOP/s of Half2's products and 280-350 of Bf16x3's, where the fp32 matrix instructions make 155.
//
// Every wave loads and splits its own rows of A, in the lanes that multiply them; B's rows are split by one wave
// and handed to the others through LDS, in 16-byte units of 8 k of one row, [plane][k-chunk][row], so that a fragment is one
// ds_read_b128.  An operand that is contiguous along its rows instead of along k is transposed in registers on the way: a lane's load of T
// neighbouring rows is a row of each of T tiles.  Splitting takes 7 vector instructions per two numbers (Half2; 21 cycles, 32
// with v_fma_mixlo_f16, which take 8 each) or 11 (Bf16x3), between the matrix instructions of the step before (the order
// is pinned: left to itself the compiler sinks the loads behind the products, and every step waits for memory).
// While a wave multiplies it goes before the other on its SIMD (s_setprio), which then prepares its next step or waits: of two waves that take turns
// by instruction neither keeps the matrix pipe busy.  32768 x 256, K = 1024 70.2 -> 67.0 us (with B's rows as columns 73.9 -> 69.7), x^T y
// 1024 x 256, K = 32768 80.3 -> 77.5, the loss's gradients of 32768 words and tokens, 256 3.20 and 3.40 -> 3.09 and 3.24 ms, 128
// 1.67 and 1.54 -> 1.48 and 1.49.  Where B's rows are kept the SIMD's second wave goes first: 32768 x 1024, K = 256 68.0 -> 65.3 (66.0 with
// both alike), the loss 2.44 -> 2.29 ms.
#include "fwp_common.hpp"
#include "fwp_gemm_plan.hpp"
#include "fwp_mfma.hpp"

#include <algorithm>
#include <type_traits>

namespace fwp {

typedef float v2f __attribute__((ext_vector_type(2)));
__device__ v2f llvm_raw_buffer_load_v2f32(v4i rsrc, int voffset, int soffset, int aux) __asm("llvm.amdgcn.raw.buffer.load.v2f32");

namespace {

typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// Registers are spilled in rare code first
__device__ __forceinline__ bool rarely(bool x) { return __builtin_expect(x, false); }
constexpr int kThreads = 256;
constexpr unsigned kOut = 0x80000000u;      // an offset beyond every buffer: reads as zero
// Offsets within a buffer are 32 bits: floats between operands' rows (Kept: up to 128 rows of B or 256 of k; kOut stays beyond), and between those of
// results (at most 64 to a wave)
constexpr int64_t kMaxLd = kMatmulMaxLd, kMaxPitch = 1 << 22;
static_assert((255 * kMaxLd + 256) * 4 <= kOut && 64 * kMaxPitch * 4 < (int64_t)1 << 32, "offsets within a tile fit 32 bits");

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

template <int P, int ROWS>
struct Planes {
    v4u u[P][kBK / 8][ROWS];
};

// The place of a row's unit in its k-chunk, such that no access meets a bank twice: a read takes lanes 0-3, 12-15, 20-23
// and 24-27 together (two chunks' rows: whole groups of four, whichever chunk), a write eight lanes, which hold two rows x
// four chunks (operands contiguous along k) or every other of sixteen rows (the others).  With rows in order and the
// chunks 32 bytes apart 420 of 1280 LDS cycles per tile step (x W^T), 770 of 1560 (g^T x) were conflicts; 32768 x 256,
// K = 1024: 4.7e7 -> 4.3e7 cycles of busy CUs, 95.0 -> 92.9 us.
__device__ __forceinline__ constexpr int unit_of(int row, int chunk) { return row ^ (2 * chunk) ^ ((row >> 3) & 3); }

// exp(x): 2^(x log2 e) by the hardware, x log2 e rounded to its nearest float and the rest of it as a factor: probabilities
// are off by at most 4 roundings, down to e^-70 (with x log2 e alone by 60 there; PyTorch's, through the logarithm, by 69).  Arguments below -150 give
// 0 as that one does (the rest of an infinity would be NaN); a NaN stays.
// exp_of_sum: 0 for a NaN, for logits whose sum of exponentials shows it.
__device__ __forceinline__ float exp_above(float x) {
    constexpr float kLog2e = 1.44269504f, kLog2eRest = 1.92596299e-8f, kLn2 = 0.693147181f;
    const float y = x * kLog2e, rest = fmaf(x, kLog2e, -y), e = __builtin_amdgcn_exp2f(y);
    return fmaf(e, fmaf(rest, kLn2, x * (kLog2eRest * kLn2)), e);
}
__device__ __forceinline__ float exp_of(float x) { return exp_above(x < -150.f ? -150.f : x); }
__device__ __forceinline__ float exp_of_sum(float x) { return exp_above(__builtin_fmaxf(x, -150.f)); }

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
    t.scaled = s.x > -INFINITY ? s.y * t.g : NAN;
    return t;
}


// The k of element e of the 8 that a lane (A) or a unit in LDS (B) holds of k-chunk c of a step: two runs of four, so that
// the four chunks' loads of one run are 64 bytes of a row.
__device__ __forceinline__ constexpr int k_of(int c, int e) { return e < 4 ? 4 * c + e : 16 + 4 * c + (e - 4); }

// Sizes of scaled elements.  Beyond kLargest they do not fit fp16.  From 2^-2 on two fp16 numbers hold them to 2^-23 of themselves, at
// kSmall to 2^-19: what is left of smaller ones is multiplied apart (add_rests), the whole of those below kTiny, fp16's smallest normal
// number (products with others cut the sum they are added to at 2^-24 of what that number would give).  With one below kLeast that is
// not enough either.
constexpr float kLargest = 65504.f, kSmall = 0x1p-6f, kTiny = 0x1p-14f, kLeast = 0x1p-31f;
// One wave's small elements at one place of a step's k cost a workgroup of the step by step kernels about as much as four steps gain over Bf16x3
// (a = 1.5 as above: 103 us, 120 when counted as one): the steps owed, beyond kGrace of them the rest of k is Bf16x3's.
constexpr int kPatience = 4, kGrace = 16;

// x = h + m (+ l) for eight values.  Half2: two fp16 numbers of x * scale; Bf16x3: three bf16 numbers of x.
struct Half2 {
    typedef _Float16 frag __attribute__((ext_vector_type(8)));
    static constexpr int kPlanes = 2;
    static constexpr bool kScaled = true;
    static __device__ __forceinline__ unsigned pack(float a, float b) {
        unsigned r;
        asm("v_cvt_pk_f16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
        return r;
    }
    static __device__ __forceinline__ void split2(float a, float b, float scale, unsigned *d) {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        d[0] = pack(a * scale, b * scale);
        const h2 h = __builtin_bit_cast(h2, d[0]);
        d[1] = pack(fmaf(a, scale, -(float)h[0]), fmaf(b, scale, -(float)h[1]));
    }
    // what is left of an element (scaled)
    static __device__ __forceinline__ float rest(float x) {
        const float h = (float)(_Float16)x, r = x - h;
        return fabsf(h) < kTiny ? x : r - (float)(_Float16)r;
    }
    // the two numbers of elements below kTiny become zero
    static __device__ __forceinline__ void drop_tiny(v4u *d) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const unsigned keep = (d[0][j] & 0x7c00u ? 0xffffu : 0u) | (d[0][j] & 0x7c000000u ? 0xffff0000u : 0u);
            d[0][j] &= keep, d[1][j] &= keep;
        }
    }
    static __device__ __forceinline__ v4f mma(frag x, frag y, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(x, y, c, 0, 0, 0); }
    // the planes (of A, of B) that are multiplied, in this order
    static constexpr int kProducts = 3;
    static constexpr int kOrder[3][2] = {{1, 0}, {0, 1}, {0, 0}};
};

// The same with the second number 2^11 times as large: its products are summed apart, and elements from 2^-16 on (of a row's largest
// in [2^14, 2^15)) are held to 2^-20 of themselves.
struct WideHalf2 : Half2 {
    static constexpr float kRest = 0x1p-11f;      // what those sums are multiplied with
    static constexpr float kLeast = 0x1p-16f;
    static __device__ __forceinline__ void split2(float a, float b, float scale, unsigned *d) {
        typedef _Float16 h2 __attribute__((ext_vector_type(2)));
        d[0] = pack(a * scale, b * scale);
        const h2 h = __builtin_bit_cast(h2, d[0]);
        d[1] = pack(fmaf(a, scale, -(float)h[0]) / kRest, fmaf(b, scale, -(float)h[1]) / kRest);
    }
};

struct Bf16x3 {
    typedef __bf16 frag __attribute__((ext_vector_type(8)));
    static constexpr int kPlanes = 3;
    static constexpr bool kScaled = false;
    static __device__ __forceinline__ void split2(float a, float b, float, unsigned *d) {
        d[0] = pack2(a, b);
        const float ra = a - low_f(d[0]), rb = b - high_f(d[0]);
        d[1] = pack2(ra, rb);
        d[2] = pack2(ra - low_f(d[1]), rb - high_f(d[1]));
    }
    static __device__ __forceinline__ v4f mma(frag x, frag y, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0); }
    static constexpr int kProducts = 6;
    static constexpr int kOrder[6][2] = {{2, 0}, {0, 2}, {1, 1}, {1, 0}, {0, 1}, {0, 0}};
};

// Elements 2 j and 2 j + 1 of eight values, split, into their place in a fragment of each plane.
template <class S>
__device__ __forceinline__ void split_pair(const float *x, int j, float scale, v4u *d) {
    unsigned y[S::kPlanes];
    S::split2(x[2 * j], x[2 * j + 1], scale, y);
#pragma unroll
    for (int p = 0; p < S::kPlanes; p++) d[p][j] = y[p];
}

// The largest and the smallest magnitude of eight elements that are not NaN.  By hand: fmaxf() and fminf() quiet every operand first, 104
// instead of 40 instructions a step.
__device__ __forceinline__ float abs_max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float abs_min3(float a, float b, float c) {
    float r;
    asm("v_min3_f32 %0, |%1|, |%2|, |%3|" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float abs_max8(const float *x) {
    return abs_max3(abs_max3(x[0], x[1], x[2]), abs_max3(x[3], x[4], x[5]), abs_max3(x[6], x[7], x[7]));
}
__device__ __forceinline__ float abs_min8(const float *x) {
    return abs_min3(abs_min3(x[0], x[1], x[2]), abs_min3(x[3], x[4], x[5]), abs_min3(x[6], x[7], x[7]));
}
// the same of those that are not zero, to one unit of the last place (NaN: all are zero)
__device__ __forceinline__ float nonzero_min8(const float *x) {
    unsigned m = ~0u;
#pragma unroll
    for (int e = 0; e < 8; e++) m = min(m, (__float_as_uint(x[e]) << 1) - 1);
    return __uint_as_float(m >> 1);
}
__device__ __forceinline__ float pick(const float *x, int e) {      // x[e] of a wave-uniform e, in registers
    typedef float v8f __attribute__((ext_vector_type(8)));
    const v8f v = {x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]};
    return v[e];
}

// A row's scale: the power of two that takes its largest element so far into [2^13, 2^14).
struct Scale {
    static constexpr unsigned kNone = 254u << 23;      // 2^127: no element but zeros yet, or below 2^-111
    float s, first;                                    // first: the largest s so far
    __device__ __forceinline__ void none() { s = __uint_as_float(kNone); }
    __device__ __forceinline__ void one() { s = 1.f; }
    __device__ __forceinline__ int exponent() const { return 127 - (int)(__float_as_uint(s) >> 23); }      // of 1 / s
    // top: 14 where no larger element can come
    __device__ __forceinline__ void set(float largest, int top = 13) {
        s = __uint_as_float((unsigned)min(254 + top - (int)(__float_as_uint(largest) >> 23), 254) << 23);
    }
    // for a row with an element of size `largest`: what its results so far are multiplied with
    __device__ __forceinline__ float fit(float largest) {
        if (!(largest * s > kLargest)) return 1.f;
        const unsigned was = __float_as_uint(s);
        set(largest);
        if (was == kNone) first = s;
        return ldexpf(1.f, (int)(__float_as_uint(s) >> 23) - (int)(was >> 23));
    }
    // s was once so much larger that the row's results so far may not be what fp32 holds
    __device__ __forceinline__ bool shrunk() const { return __float_as_uint(s) != kNone && s < first * 0x1p-25f; }
};

__device__ __forceinline__ void drop_tiny8(float *x, float s) {
#pragma unroll
    for (int e = 0; e < 8; e++) x[e] = fabsf((float)(_Float16)(x[e] * s)) < kTiny ? 0.f : x[e];
}

// A lane's elements of ROWS rows, scaled: the largest magnitude, and each row's before that; the smallest; the smallest that is not zero, which takes
// three times the instructions: looked for from the first zero on (32768 x 256, K = 1024 always 72.4 us, so 71.1; where a zero of B's rows, beyond the last
// of 776, led to a second look at every step, 8192 x 776, K = 1024 70.1 -> 62.9).
template <int ROWS>
__device__ __forceinline__ float largest_of(const float (&x)[ROWS][8], const Scale (&s)[ROWS], float (&m)[ROWS]) {
    float all = 0.f;
#pragma unroll
    for (int i = 0; i < ROWS; i++) m[i] = abs_max8(x[i]), all = abs_max3(all, m[i] * s[i].s, 0.f);
    return all;
}
template <int ROWS>
__device__ __forceinline__ float smallest_of(const float (&x)[ROWS][8], const Scale (&s)[ROWS]) {
    float all = INFINITY;
#pragma unroll
    for (int i = 0; i < ROWS; i++) all = abs_min3(all, abs_min8(x[i]) * s[i].s, INFINITY);
    return all;
}
template <int ROWS>
__device__ __forceinline__ float smallest_nonzero_of(const float (&x)[ROWS][8], const Scale (&s)[ROWS]) {
    float all = INFINITY;
#pragma unroll
    for (int i = 0; i < ROWS; i++) all = abs_min3(all, nonzero_min8(x[i]) * s[i].s, INFINITY);
    return all;
}
// Which of the wave's lanes' elements are small (bit e: those at e; bit 8: some are tiny); far: one is too small even for its rest.  Two
// instructions an element: with gradients as operands it is run every few steps (a loop over e that picks the elements: 10 an element, a training step of the
// benchmark's model 0.3 ms more).
constexpr unsigned kSomeTiny = 1u << 8;
template <int ROWS>
__device__ __forceinline__ unsigned small_of(const float (&x)[ROWS][8], const Scale (&s)[ROWS], bool &far) {
    const float least = smallest_nonzero_of(x, s);
    if (!__any(least < kSmall)) return 0;
    far |= least < kLeast;
    unsigned m = __any(least < kTiny) ? kSomeTiny : 0u, below[ROWS];      // below: twice the bits of kSmall / s, as a zero's are largest
#pragma unroll
    for (int i = 0; i < ROWS; i++) below[i] = (__float_as_uint(ldexpf(kSmall, s[i].exponent())) << 1) - 1;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        bool small = false;
#pragma unroll
        for (int i = 0; i < ROWS; i++) small |= (__float_as_uint(x[i][e]) << 1) - 1 < below[i];
        m |= __any(small) ? 1u << e : 0u;
    }
    return m;
}

// LDS accesses of one wave execute in order; this keeps the compiler from moving them across.
__device__ __forceinline__ void wave_lds_order() { asm volatile("" ::: "memory"); }

// A: a wave's 16 T rows, straight from global memory to the lanes that multiply them.  Lane 16 c + r holds k-chunk c of
// row r of each of the T matrix-instruction tiles; a tile's rows are 16 consecutive ones (KC: rows are contiguous along
// k) or every T-th of 16 T (contiguous along the rows: a lane's load is T neighbouring rows).
// NLL: the operand is the loss gradient, formed from the logits; tokens are the rows (KC) or k.
template <bool KC, int T, bool NLL>
struct Direct {
    // a step's elements as they are loaded, and (NLL, !KC) one of its 32 tokens
    struct Raw {
        float x[T][8];
        NllToken next;
    };
    NllToken token[NLL && KC ? T : 1];
    NllToken *tok;      // LDS, this wave's: a step's tokens
    Scale s[T];
    int c, r;
    unsigned at[2];

    static __device__ __forceinline__ int row_of(int i, int r) { return KC ? 16 * i + r : T * r + i; }

    __device__ __forceinline__ void init(int lane, int row0, int rows, const NllArgs &nll) {
        c = lane / 16, r = lane % 16;
        if constexpr (NLL && KC)
#pragma unroll
            for (int i = 0; i < T; i++) token[i] = nll_token(nll, min(row0 + row_of(i, r), rows - 1));
    }
    // the lanes' offsets for a load of k0 ...: they change where a row ends within the step only
    __device__ __forceinline__ void aim(int64_t ld, int k0, int K) {
        if constexpr (KC) {
            const unsigned o = (unsigned)(r * ld + 4 * c) * 4;
            at[0] = k0 + 4 * c < K ? o : kOut, at[1] = k0 + 16 + 4 * c < K ? o + 64 : kOut;
        } else {
            at[0] = (unsigned)(4 * c * ld + T * r) * 4;
        }
    }
    // P: the wave's first row at k = 0, `left` rows from there, k0 .. min(k0 + kBK, K); zeros beyond K
    __device__ __forceinline__ void load(Raw &w, const float *P, int64_t ld, int left, int k0, int K, const NllArgs &nll, int tokens,
                                         int lane) const {
        if constexpr (KC) {
            const v4i rs = buffer_of(P + k0, k0 < K && left > 0 ? (int64_t)(min(left, 16 * T) - 1) * ld + (K - k0) : 0);
#pragma unroll
            for (int i = 0; i < T; i++) {
                const v4f a = llvm_raw_buffer_load_v4f32(rs, (int)at[0], (int)(i * ld * 64), 0),
                          b = llvm_raw_buffer_load_v4f32(rs, (int)at[1], (int)(i * ld * 64), 0);
#pragma unroll
                for (int j = 0; j < 4; j++) w.x[i][j] = a[j], w.x[i][4 + j] = b[j];
            }
        } else {
            const int64_t size = (int64_t)(min(K - k0, kBK) - 1) * ld + left;
            const v4i rs = buffer_of(P + (int64_t)k0 * ld, k0 < K && size > 0 ? size : 0);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int so = (int)(k_of(0, e) * ld * 4);
                if constexpr (T == 2) {
                    const v2f a = llvm_raw_buffer_load_v2f32(rs, (int)at[0], so, 0);
                    w.x[0][e] = a[0], w.x[1][e] = a[1];
                } else {
                    static_assert(T == 1, "one or two rows per load");
                    w.x[0][e] = llvm_raw_buffer_load_f32(rs, (int)at[0], so, 0);
                }
            }
            if constexpr (NLL) w.next = nll_token(nll, min(k0 + lane % kBK, tokens - 1));
        }
    }
    // zeros beyond K (a row contiguous along k runs on into the next row there)
    __device__ __forceinline__ void cut(Raw &w, int k0, int K) const {
        if constexpr (KC)
#pragma unroll
            for (int i = 0; i < T; i++)
#pragma unroll
                for (int e = 0; e < 8; e++) w.x[i][e] = k0 + k_of(c, e) < K ? w.x[i][e] : 0.f;
    }
    // the step's tokens to where element() reads them
    __device__ __forceinline__ void hand_over(const Raw &w, int lane) const {
        if constexpr (NLL && !KC) {
            wave_lds_order();
            if (lane < kBK) tok[lane] = w.next;
            wave_lds_order();
        }
    }
    // the operand's element: itself, or the loss gradient in place of the logit; `whole`: also where a target or K's end is
    // within the step (rare())
    __device__ __forceinline__ float element(const Raw &w, int i, int e, bool whole, int row0, int k0, int K) const {
        if constexpr (!NLL) return w.x[i][e];
        else {
            const NllToken t = KC ? token[i] : tok[k_of(c, e)];
            if (!whole) return exp_of_sum(w.x[i][e] - t.shift) * t.scaled;
            const int k = k0 + k_of(c, e);
            // a token beyond K has the last one's values beside a logit of 0: its exponential may be infinite
            const float d = fmaf(exp_of(w.x[i][e] - t.shift), t.scaled, t.hit == (KC ? k : row0 + row_of(i, r)) ? -t.g : 0.f);
            return k < K ? d : 0.f;
        }
    }
    __device__ __forceinline__ bool rare(const Raw &w, int row0, int k0, int K) const {
        if constexpr (!NLL) return false;
        bool any = k0 + kBK > K;
        if constexpr (!KC) any |= (unsigned)(w.next.hit - row0) < 16 * T;
        else
#pragma unroll
            for (int i = 0; i < T; i++) any |= (unsigned)(token[i].hit - k0) < kBK;
        return __any(any);
    }
    // the largest magnitude of a row in this step from its lanes' own
    static __device__ __forceinline__ float of_row(float m) {
        m = fmaxf(m, __shfl_xor(m, 16, 64));
        return fmaxf(m, __shfl_xor(m, 32, 64));
    }
};

// B: a thread's share of the loads of a workgroup's ROWS rows and of their split parts' LDS writes.  KC: a task is one
// k-chunk of one row; otherwise of VEC neighbouring rows.  A row's four k-chunks are in one wave.
template <bool KC, int ROWS, int WAVES>
struct Staged {
    static constexpr int kUnits = ROWS / (16 * WAVES);
    static constexpr int VEC = KC ? 1 : kUnits;
    struct Raw {
        float x[kUnits][8];
    };
    Scale s[kUnits];
    int c, r, unit;
    unsigned at[2];

    __device__ __forceinline__ void init(int tid) {
        c = KC ? tid % 4 : tid % 64 / 16;
        r = KC ? tid / 4 : (tid / 64 * 16 + tid % 16) * VEC;
        unit = c * ROWS + unit_of(r, c);
    }
    __device__ __forceinline__ int row_of(int t) const { return KC ? r + 16 * WAVES * t : r + t; }
    __device__ __forceinline__ void aim(int64_t ld, int k0, int K) {
        if constexpr (KC) {
            const unsigned o = (unsigned)(r * ld + 4 * c) * 4;
            at[0] = k0 + 4 * c < K ? o : kOut, at[1] = k0 + 16 + 4 * c < K ? o + 64 : kOut;
        } else {
            at[0] = (unsigned)(4 * c * ld + r) * 4;
        }
    }
    __device__ __forceinline__ void load(Raw &w, const float *P, int64_t ld, int left, int k0, int K) const {
        if constexpr (KC) {
            const v4i rs = buffer_of(P + k0, k0 < K ? (int64_t)(min(left, ROWS) - 1) * ld + (K - k0) : 0);
#pragma unroll
            for (int t = 0; t < kUnits; t++) {
                const v4f a = llvm_raw_buffer_load_v4f32(rs, (int)at[0], (int)(t * ld * 64 * WAVES), 0),
                          b = llvm_raw_buffer_load_v4f32(rs, (int)at[1], (int)(t * ld * 64 * WAVES), 0);
#pragma unroll
                for (int j = 0; j < 4; j++) w.x[t][j] = a[j], w.x[t][4 + j] = b[j];
            }
        } else {
            const v4i rs = buffer_of(P + (int64_t)k0 * ld, k0 < K ? (int64_t)(min(K - k0, kBK) - 1) * ld + left : 0);
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int so = (int)(k_of(0, e) * ld * 4);
                if constexpr (VEC == 2) {
                    const v2f a = llvm_raw_buffer_load_v2f32(rs, (int)at[0], so, 0);
                    w.x[0][e] = a[0], w.x[1][e] = a[1];
                } else {
                    static_assert(VEC == 1, "one or two rows per load");
                    w.x[0][e] = llvm_raw_buffer_load_f32(rs, (int)at[0], so, 0);
                }
            }
        }
    }
    __device__ __forceinline__ void cut(Raw &w, int k0, int K) const {
        if constexpr (KC)
#pragma unroll
            for (int t = 0; t < kUnits; t++)
#pragma unroll
                for (int e = 0; e < 8; e++) w.x[t][e] = k0 + k_of(c, e) < K ? w.x[t][e] : 0.f;
    }
    static __device__ __forceinline__ float of_row(float m) {
        m = fmaxf(m, __shfl_xor(m, KC ? 1 : 16, 64));
        return fmaxf(m, __shfl_xor(m, KC ? 2 : 32, 64));
    }
    // the wave that splits the rows of matrix-instruction tile j
    static constexpr int owner(int j) { return KC ? j % WAVES : j / VEC; }
    // a unit's split parts to LDS
    template <int P>
    __device__ __forceinline__ void store(Planes<P, ROWS> &L, int t, const v4u *d) const {
#pragma unroll
        for (int p = 0; p < P; p++) L.u[p][0][KC ? unit + 16 * WAVES * t : unit ^ t] = d[p];
    }
    // fp32 as it is: 16-byte units of a chunk's four k, [chunk][half][row]
    __device__ __forceinline__ void store_plain(v4f *L, const Raw &w) const {
#pragma unroll
        for (int t = 0; t < kUnits; t++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                L[(2 * c + h) * ROWS + row_of(t)] = v4f{w.x[t][4 * h], w.x[t][4 * h + 1], w.x[t][4 * h + 2], w.x[t][4 * h + 3]};
    }
};

struct GemmArgs {
    const float *A, *B;
    float *C;                    // the result, or (several k ranges) one M x N partial result per range, `part` floats apart
    int64_t lda, ldb, ldc, part;
    int M, N, K;
    int ks;                      // k per range (a multiple of kBK)
    int vec;                     // C, residual and gate lie 16-byte aligned, in rows of whole 16-byte groups
    int tm, tn, ranges;          // tiles, of k
    float *colsum;               // sums over k of A's rows, per range [M] (A contiguous along its rows), or NULL
    fwp_mm_epilogue epi;         // applied here when there is one range
    NllArgs nll;
    // per tile of columns and row: the largest logit and the sum of exp(logit - largest); logits of the targets
    float *part_max, *part_sum, *hit;
    v4u *image;                  // B split, as k_image leaves it, or NULL
};

enum { kPlain = 0, kLse = 1, kGrad = 2 };

// everything but the bias
__device__ __forceinline__ float apply(const fwp_mm_epilogue &e, float x, int64_t at) {
    if (e.relu) x = relu(x);
    if (e.residual) x += e.residual[at];
    if (e.gate) x = gated(e.gate[at], x);
    return x;
}

// What a sum of exp(logit - m) is multiplied with to become one of exp(logit - big).  A part of the vocabulary with no
// logit but -infinity (masked words; columns beyond the last) has m = -infinity and the sum 0, or NaN if there
// was one: it stays as it is (exp(-infinity + infinity) would make it NaN).
__device__ __forceinline__ float to_max(float m, float big) { return m == -INFINITY ? 1.f : exp_of(m - big); }

// What becomes of a column of results on its way out (LDS): 2^exponent, the bias.
struct Columns {
    const int *exponent;
    const float *bias;
};

// acc[i][j][r] is row m0 + row[i], column n0 + 16 j + 4 lc + r, scaled: B's rows are the rows of the matrix instructions'
// results, so that a lane has four neighbouring columns of a row, 16 bytes.  `rows`: those of the wave.  The two scales are taken
// back in one step: one alone can leave fp32's range where both together do not.
template <bool SCALED, int MT, int NT, int MODE>
__device__ __forceinline__ void finish(const GemmArgs &g, v4f (&acc)[MT][NT], const int (&row)[MT], int m0, int rows, int n0, int lc,
                                       const int (&ea)[MT], const Columns &col, int range, int column_tile) {
    const bool one = g.ranges == 1;
    const int left = min(g.M - m0, rows), nl = g.N - n0;
    if (left <= 0) return;
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const v4f b = *reinterpret_cast<const v4f *>(col.bias + 16 * j + 4 * lc);
        v4i eb = {0, 0, 0, 0};
        if constexpr (SCALED) eb = *reinterpret_cast<const v4i *>(col.exponent + 16 * j + 4 * lc);
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[i][j][e] = (SCALED ? ldexpf(acc[i][j][e], ea[i] + eb[e]) : acc[i][j][e]) + b[e];
    }
    const int64_t first = (int64_t)m0 * g.ldc + n0, size = (int64_t)(left - 1) * g.ldc + nl;
    float *const C = g.C + range * g.part + first;
    if (MODE == kLse && !g.C) {
    } else if (nl >= 16 * NT && g.ldc <= kMaxPitch) {
        // Rows beyond M lie behind the resource.  Buffer accesses need 4-byte alignment only, whatever N is (32768 x 1029, K = 256 74 us, element by
        // element 116).
        unsigned at[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) at[i] = (unsigned)(row[i] * g.ldc + 4 * lc) * 4;
        if (one && g.epi.relu)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[i][j][e] = relu(acc[i][j][e]);
        // a tile's loads all at once: one by one, each waited for, they bound the product
        const auto with = [&](const float *P, auto f) {
            const v4i rs = buffer_of(P + first, size);
#pragma unroll
            for (int i = 0; i < MT; i++) {
                v4f y[NT];
#pragma unroll
                for (int j = 0; j < NT; j++) y[j] = llvm_raw_buffer_load_v4f32(rs, (int)(at[i] + 64 * j), 0, 0);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[i][j][e] = f(acc[i][j][e], y[j][e]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (one && g.epi.residual) with(g.epi.residual, [](float x, float y) { return x + y; });
        if (one && g.epi.gate) with(g.epi.gate, [](float x, float y) { return gated(y, x); });
        const v4i rs = buffer_of(C, size);
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int i = 0; i < MT; i++) llvm_raw_buffer_store_v4f32(acc[i][j], rs, (int)(at[i] + 64 * j), 0, 0);
    } else {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const int n = 16 * j + 4 * lc;
                const int64_t at = row[i] * g.ldc + n;
                if (row[i] >= left || n >= nl) continue;
                v4f v = acc[i][j];
                if (g.vec) {
                    if (one) {
                        if (g.epi.relu) v = v4f{relu(v[0]), relu(v[1]), relu(v[2]), relu(v[3])};
                        if (g.epi.residual) v += *reinterpret_cast<const v4f *>(g.epi.residual + first + at);
                        if (g.epi.gate) {
                            const v4f y = *reinterpret_cast<const v4f *>(g.epi.gate + first + at);
                            v = v4f{gated(y[0], v[0]), gated(y[1], v[1]), gated(y[2], v[2]), gated(y[3], v[3])};
                        }
                    }
                    *reinterpret_cast<v4f *>(C + at) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (n + e < nl) C[at + e] = one ? apply(g.epi, v[e], first + at + e) : v[e];
                }
            }
    }
    if constexpr (MODE == kLse) {
        // the largest of a row's logits here and the sum of exp(logit - largest); four lanes share a row
        if (nl < 16 * NT)
#pragma unroll
            for (int j = 0; j < NT; j++)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (16 * j + 4 * lc + e >= nl)
#pragma unroll
                        for (int i = 0; i < MT; i++) acc[i][j][e] = -INFINITY;
#pragma unroll
        for (int i = 0; i < MT; i++) {
            const int m = m0 + row[i];
            if (g.hit) {
                const int at = row[i] < left ? (int)g.nll.target[m] - n0 - 4 * lc : -1;
#pragma unroll
                for (int j = 0; j < NT; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        if (at == 16 * j + e && at + 4 * lc < nl) g.hit[m] = acc[i][j][e];
            }
            float big = -INFINITY, s = 0.f;
#pragma unroll
            for (int j = 0; j < NT; j++) big = fmaxf(fmaxf(big, fmaxf(acc[i][j][0], acc[i][j][1])), fmaxf(acc[i][j][2], acc[i][j][3]));
            big = fmaxf(big, __shfl_xor(big, 16, 64));
            big = fmaxf(big, __shfl_xor(big, 32, 64));
            const float z = big == -INFINITY ? 0.f : big;
#pragma unroll
            for (int j = 0; j < NT; j++) s += (exp_of(acc[i][j][0] - z) + exp_of(acc[i][j][1] - z)) + (exp_of(acc[i][j][2] - z) + exp_of(acc[i][j][3] - z));
            s += __shfl_xor(s, 16, 64);
            s += __shfl_xor(s, 32, 64);
            if (lc == 0 && row[i] < left) {
                const int64_t at = (int64_t)column_tile * g.M + m;
                g.part_max[at] = big, g.part_sum[at] = s;
            }
        }
    }
}

// What two fp16 numbers leave of small elements, in fp32: the step's products of the rest of A with B and of A with the rest of B, for
// the k of bit e of `small_a` (a wave's rows) and of `small_b`.  x, f: the step's elements of A, split.  has, rest: whether column tile j has a
// rest at e, and this lane's of it.
template <int MT, int NT, class Has, class Rest>
__device__ __forceinline__ void add_rests(v4f (&acc)[MT][NT], const float (&x)[MT][8], const Scale (&s)[MT], unsigned small_a, unsigned small_b,
                                          v4u (&f)[MT][Half2::kPlanes], const Planes<Half2::kPlanes, 16 * NT> &L, const int (&unit)[2], Has has, Rest rest) {
    if (small_a & kSomeTiny)
#pragma unroll
        for (int i = 0; i < MT; i++) Half2::drop_tiny(f[i]);
#pragma unroll 1
    for (unsigned left = (small_a | small_b) & 0xff; left; left &= left - 1) {
        const int e = __builtin_ctz(left);
        float v[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) v[i] = pick(x[i], e) * s[i].s;
        if (small_b >> e & 1)
#pragma unroll
            for (int j = 0; j < NT; j++)
                if (has(j, e)) {
                    const float y = rest(j, e);
#pragma unroll
                    for (int i = 0; i < MT; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(y, v[i], acc[i][j], 0, 0, 0);
                }
        if (small_a >> e & 1) {
#pragma unroll
            for (int i = 0; i < MT; i++) v[i] = Half2::rest(v[i]);
#pragma unroll
            for (int j = 0; j < NT; j++) {
                const _Float16 *const h = reinterpret_cast<const _Float16 *>(&L.u[0][0][unit[j % 2] + 16 * j]) + e;
                const float y = (float)h[0] + (float)h[sizeof(L.u[0]) / sizeof(_Float16)];
#pragma unroll
                for (int i = 0; i < MT; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(y, v[i], acc[i][j], 0, 0, 0);
            }
        }
    }
}

// The same for A alone with whole steps of 16-bit products: small elements leave f and come back 2^20 times as large, those that are small then 2^40
// times, to results as much larger meanwhile (below 2^(28 + 8) before, K <= 256).  Each is the step's products once more, however many elements:
// 32768 x 1024, K = 256, features of sizes exp(a N(0,1)), a = 0 / 1.5 / 3 / 5 66 / 74 / 128 / 140 us (Bf16x3 97; element by element 68 / 76 / 183 / 581).
constexpr float kLevel = 0x1p20f, kFarthest = 0x1p-50f;
template <int MT, int NT>
__device__ __forceinline__ void add_small(v4f (&acc)[MT][NT], const float (&x)[MT][8], const Scale (&s)[MT], v4u (&f)[MT][Half2::kPlanes],
                                          const Planes<Half2::kPlanes, 16 * NT> &L, const int (&unit)[2]) {
    typedef Half2 S;
    const float least = smallest_nonzero_of(x, s);
    // elements of row tile i of sizes (scaled) from `from` below `to` (also infinities: infinity), times up
    const auto part = [&](int i, float from, float to, float up, v4u *d) {
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float y[2];
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const float v = x[i][2 * j + e] * s[i].s;
                y[e] = fabsf(v) < from || (to < INFINITY && fabsf(v) >= to) ? 0.f : v;
            }
            unsigned w[S::kPlanes];
            S::split2(y[0], y[1], up, w);
#pragma unroll
            for (int p = 0; p < S::kPlanes; p++) d[p][j] = w[p];
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int i = 0; i < MT; i++) {
        part(i, kSmall, INFINITY, 1.f, f[i]);
        float to = kSmall, up = 1.f;
#pragma unroll 1
        do {
            const float from = to / kLevel;
            v4u d[S::kPlanes];
            up *= kLevel;
            part(i, from, to, up, d);
#pragma unroll
            for (int j = 0; j < NT; j++) {
                acc[i][j] *= kLevel;
#pragma unroll
                for (int q = 0; q < S::kProducts; q++)
                    acc[i][j] = S::mma(__builtin_bit_cast(S::frag, L.u[S::kOrder[q][1]][0][unit[j % 2] + 16 * j]),
                                       __builtin_bit_cast(S::frag, d[S::kOrder[q][0]]), acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
            }
            to = from;
        } while (__any(least < to));
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] *= 1.f / up;
    }
}

// B split into Bf16x3's numbers: [tile of BN columns][step of k] the step's place in LDS as it is, zeros beyond K.  A workgroup a step.
static_assert(Bf16x3::kPlanes == kImagePlanes, "the image's size");
template <int BN>
__global__ __launch_bounds__(2 * BN) void k_image(const float *__restrict__ B, int64_t ldb, int N, int K, v4u *__restrict__ image) {
    typedef Planes<Bf16x3::kPlanes, BN> Stage;
    const int k0 = blockIdx.x * kBK, n0 = blockIdx.y * BN;
    Staged<false, BN, BN / 32> b;
    typename Staged<false, BN, BN / 32>::Raw x;
    b.init(threadIdx.x);
    b.aim(ldb, k0, K);
    b.load(x, B + n0, ldb, N - n0, k0, K);
    Stage &to = reinterpret_cast<Stage *>(image)[(int64_t)blockIdx.y * gridDim.x + blockIdx.x];
#pragma unroll
    for (int t = 0; t < b.kUnits; t++) {
        v4u part[Bf16x3::kPlanes];
#pragma unroll
        for (int j = 0; j < 4; j++) split_pair<Bf16x3>(x.x[t], j, 1.f, part);
        b.store(to, t, part);
    }
}

// A workgroup of WAVES waves: a wave 16 MT rows and all 16 NT columns; B's rows are staged step by step, in two
// alternating places, one barrier a step; IMAGE: they come split.  What bounds it: 32768 x 256, K = 1024 takes 71 us (one 128 x 128 tile with both
// operands through LDS, Bf16x3: 89): products alone 36 us, the split 10 us, loads 8, LDS 6, the look for small elements 7.
template <class S, bool AKC, bool BKC, int MT, int NT, int MODE, int WAVES = 4, bool IMAGE = false>
__global__ __launch_bounds__(64 * WAVES, 2) void k_gemm(GemmArgs g) {
    constexpr int WM = 16 * MT, BM = WAVES * WM, BN = 16 * NT;
    static_assert(WAVES == 4 || !S::kScaled, "four waves' changes of scales");
    static_assert(!IMAGE || !S::kScaled, "an image of Bf16x3's numbers");
    typedef Direct<AKC, MT, MODE == kGrad> OpA;
    typedef Staged<BKC, BN, WAVES> OpB;
    // the two places of a step's B, and (scaled) behind them its elements in fp32 where some are small; later Bf16x3's places
    typedef v4f Elements[2][4][BN];
    constexpr size_t kStages = 2 * sizeof(Planes<S::kPlanes, BN>), kShared = kStages + (S::kScaled ? 2 * sizeof(Elements) : 0);
    static_assert(2 * sizeof(Planes<Bf16x3::kPlanes, BN>) <= kShared, "Bf16x3's places fit");
    static_assert(sizeof(v4f) * 8 * BN <= kShared, "fp32 of a step fits");
    __shared__ __align__(16) char shared[kShared];
    __shared__ __align__(16) int exponents[BN];
    __shared__ __align__(16) float biases[BN];
    // Of the steps' B, alternately: what each wave did to its rows' scales (kChange: what their results so far are multiplied with is in
    // change_b) and which of its elements are small (bit e); of how many e there are small elements of A; whether an element is too small for that
    constexpr int kChange = 1 << 9, kStop = 1 << 10, kCountA = 1 << 12;
    __shared__ __align__(16) int news[2][4];
    __shared__ __align__(16) float change_b[S::kScaled ? 2 : 1][S::kScaled ? BN : 4];
    __shared__ float change_a[S::kScaled ? 4 : 1][WM];
    __shared__ int odd_waves[WAVES];
    __shared__ NllToken toks[MODE == kGrad && !AKC ? WAVES : 1][MODE == kGrad && !AKC ? kBK : 1];
    Elements *const scaled_b = reinterpret_cast<Elements *>(shared + kStages);
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    // workgroups go round the 8 XCDs: each XCD gets a run of neighbouring tiles (a row of tiles reads the same
    // rows of A, through that XCD's L2), of whole ranges of k where there are several: the tiles of a range read the
    // same k of A and B (2048 x 128, K = 24576 in 32 ranges: 65 us, with each XCD a tile of all ranges 74)
    const int total = gridDim.x, xcd = blockIdx.x % 8, each = total / 8, rest = total % 8;
    const int tile = xcd * each + min(xcd, rest) + blockIdx.x / 8, range = tile / (g.tm * g.tn), id = tile % (g.tm * g.tn);
    const int m0 = (id / g.tn) * BM + wave * WM, n0 = (id % g.tn) * BN;
    const int kb = range * g.ks, ke = min(g.K, kb + g.ks);
    const float *Ap = AKC ? g.A + (int64_t)m0 * g.lda : g.A + m0;
    const float *Bp = BKC ? g.B + (int64_t)n0 * g.ldb : g.B + n0;
    const int ml = g.M - m0, nl = g.N - n0;
    const int lr = lane % 16, lc = lane / 16;
    // unit_of(16 j + lr, lc) of even and odd j
    const int unit[2] = {lc * BN + unit_of(lr, lc), lc * BN + unit_of(16 + lr, lc) - 16};
    OpA a;
    OpB b;
    a.init(lane, m0, g.M, g.nll);
    b.init(tid);
    a.tok = toks[MODE == kGrad && !AKC ? wave : 0];
    const auto load = [&](typename OpA::Raw &x, typename OpB::Raw &y, int k0) {
        a.load(x, Ap, g.lda, ml, k0, ke, g.nll, g.K, lane);
        b.load(y, Bp, g.ldb, nl, k0, ke);
    };
    const auto aim = [&](int k0) { a.aim(g.lda, k0, ke), b.aim(g.ldb, k0, ke); };
    float csum[MT];
    const bool sums = !AKC && g.colsum && n0 == 0;
    v4f acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        a.s[i].none();
        csum[i] = 0.f;
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int t = 0; t < OpB::kUnits; t++) b.s[t].none();

    // IMAGE: a thread's share of a step's B
    constexpr int kStep = IMAGE ? Bf16x3::kPlanes * kBK / 8 * BN : 0, kShare = IMAGE ? kStep / (64 * WAVES) : 1;
    v4u share[kShare];
    const v4u *const image = IMAGE ? g.image + (int64_t)(n0 / BN) * ((g.K + kBK - 1) / kBK) * kStep : nullptr;
    const auto ask = [&](int k0) {
        if constexpr (IMAGE) {
            const v4i rs = buffer_of(reinterpret_cast<const float *>(image + (int64_t)(k0 / kBK) * kStep), k0 < ke ? 4 * kStep : 0);
#pragma unroll
            for (int i = 0; i < kShare; i++) share[i] = __builtin_bit_cast(v4u, llvm_raw_buffer_load_v4f32(rs, 16 * tid, i * 1024 * WAVES, 0));
        }
    };
    const auto put = [&](auto &to, int i) {
        if constexpr (IMAGE) (&to.u[0][0][0])[i * 64 * WAVES + tid] = share[i];
    };

    typename OpA::Raw ra[2];
    typename OpB::Raw rb[2];
    bool far = false;         // results that may not be what fp32 holds
    // The steps from k = first on with operands split as T; returns the k it stopped at (scaled).
    const auto steps = [&](auto split_as, int first) __attribute__((always_inline)) -> int {
        typedef decltype(split_as) T;
        typedef typename T::frag frag;
        typedef Planes<T::kPlanes, BN> Stage;
        Stage *const L = reinterpret_cast<Stage *>(shared);
        bool change = false;      // of scales of A's rows
        unsigned small_a = 0;
        bool zeros_a = false, zeros_b = false;      // there are zeros: ReLU's, rows beyond the last
        int spent = 0;
        v4u fa[2][MT][T::kPlanes];
        float part_sum[MT];       // of a step's elements of A's rows
        const auto split_a = [&](int i, int j, const typename OpA::Raw &x, v4u (*f)[T::kPlanes], bool whole, int k0) {
            float v[8];
            v[2 * j] = a.element(x, i, 2 * j, whole, m0, k0, ke), v[2 * j + 1] = a.element(x, i, 2 * j + 1, whole, m0, k0, ke);
            if constexpr (!AKC) part_sum[i] = (j ? part_sum[i] : 0.f) + (v[2 * j] + v[2 * j + 1]);
            else part_sum[i] = 0.f;
            split_pair<T>(v, j, a.s[i].s, f[i]);
        };
        // Pair q of the 4 (units + MT) pairs of a step's split: B's units first, each to LDS when it is whole, then A's tiles
        v4u part[T::kPlanes];
        constexpr int kUnits = IMAGE ? 0 : OpB::kUnits, kPairs = 4 * (kUnits + MT);
        const auto split = [&](int q, const typename OpA::Raw &x, const typename OpB::Raw &y, v4u (*f)[T::kPlanes], Stage &to, int k0) {
            if (q < 4 * kUnits) {
                split_pair<T>(y.x[q / 4], q % 4, b.s[q / 4].s, part);
                if (q % 4 == 3) b.store(to, q / 4, part);
                return;
            }
            const int j = (q - 4 * kUnits) / MT, i = q % MT;
            split_a(i, j, x, f, false, k0);
        };
        // once more where split() left something out
        const auto complete = [&](const typename OpA::Raw &x, v4u (*f)[T::kPlanes], int k0) {
            if constexpr (MODE == kGrad)
                if (a.rare(x, m0, k0, ke))
#pragma unroll
                    for (int i = 0; i < MT; i++)
#pragma unroll
                        for (int j = 0; j < 4; j++) split_a(i, j, x, f, true, k0);
        };
        // What a step's split needs: zeros beyond K, and (parity: the step's) scales that its elements fit
        const auto prepare = [&](typename OpA::Raw &x, typename OpB::Raw &y, int k0, int parity) __attribute__((always_inline)) {
            a.hand_over(x, lane);
            if (ke % 4 && k0 + kBK > ke) {
                a.cut(x, k0, ke);
                if constexpr (!IMAGE) b.cut(y, k0, ke);
            }
            if constexpr (T::kScaled) {
                float ma[MT], mb[OpB::kUnits];
                const bool beyond = fmaxf(largest_of(x.x, a.s, ma), largest_of(y.x, b.s, mb)) > kLargest;
                float la = zeros_a ? smallest_nonzero_of(x.x, a.s) : smallest_of(x.x, a.s);
            float lb = zeros_b ? smallest_nonzero_of(y.x, b.s) : smallest_of(y.x, b.s);
                int word = 0;
                small_a = 0;
                if (rarely(__any(beyond || fminf(la, lb) < kSmall))) {
                zeros_a |= __any(la == 0.f) != 0, zeros_b |= __any(lb == 0.f) != 0;
                    if (__any(beyond)) {
                        change = true, word = kChange;
                        la = lb = 0.f;
#pragma unroll
                        for (int i = 0; i < MT; i++) change_a[wave][OpA::row_of(i, lr)] = a.s[i].fit(OpA::of_row(ma[i])), far |= a.s[i].shrunk();
#pragma unroll
                        for (int t = 0; t < OpB::kUnits; t++) change_b[parity][b.row_of(t)] = b.s[t].fit(OpB::of_row(mb[t])), far |= b.s[t].shrunk();
                    }
                    bool stop = false;
                    if (__any(la < kSmall)) small_a = small_of(x.x, a.s, stop), word |= __popc(small_a) * kCountA;
                    if (__any(lb < kSmall)) word |= small_of(y.x, b.s, stop);
                    if (__any(stop)) word |= kStop;
                    if (word & 0xff)
#pragma unroll
                        for (int t = 0; t < OpB::kUnits; t++)
#pragma unroll
                            for (int h = 0; h < 2; h++)
                                scaled_b[parity][h][b.c][b.row_of(t)] =
                                    v4f{y.x[t][4 * h], y.x[t][4 * h + 1], y.x[t][4 * h + 2], y.x[t][4 * h + 3]} * b.s[t].s;
                    if (word & kSomeTiny)
#pragma unroll
                        for (int t = 0; t < OpB::kUnits; t++) drop_tiny8(y.x[t], b.s[t].s);
                }
                if (lane == 0) news[parity][wave] = word;
            }
        };
        // Before step k0's products (x: its elements of A): results so far to its scales, and what is left of its small elements
        // True (in all waves): the step is not for fp16.
        const auto follow = [&](int parity, const typename OpA::Raw &x) __attribute__((always_inline)) -> bool {
            if constexpr (T::kScaled) {
                const int4 w = *reinterpret_cast<const int4 *>(news[parity]);
                const int of[4] = {__builtin_amdgcn_readfirstlane(w.x), __builtin_amdgcn_readfirstlane(w.y), __builtin_amdgcn_readfirstlane(w.z),
                                   __builtin_amdgcn_readfirstlane(w.w)};
                const int all = of[0] | of[1] | of[2] | of[3];
                if (rarely(all & kChange)) {
#pragma unroll
                    for (int j = 0; j < NT; j++)
                        if (of[OpB::owner(j)] & kChange)
#pragma unroll
                            for (int i = 0; i < MT; i++) acc[i][j] *= *reinterpret_cast<const v4f *>(change_b[parity] + 16 * j + 4 * lc);
                }
                if (rarely(change)) {
                    change = false;
#pragma unroll
                    for (int i = 0; i < MT; i++)
#pragma unroll
                        for (int j = 0; j < NT; j++) acc[i][j] *= change_a[wave][OpA::row_of(i, lr)];
                }
                if (rarely(all & (0xff | kStop | 0xf * kCountA))) {
                    spent += kPatience * (of[0] / kCountA + of[1] / kCountA + of[2] / kCountA + of[3] / kCountA + __popc(all & 0xff));
                    if (all & kStop || spent > kGrace) return true;
                    add_rests(acc, x.x, a.s, small_a, all & 0xff, fa[parity], L[parity], unit, [&](int j, int e) { return of[OpB::owner(j)] >> e & 1; },
                              [&](int j, int e) { return Half2::rest(reinterpret_cast<const float *>(&scaled_b[parity][e / 4][lc][16 * j + lr])[e % 4]); });
                }
                spent = max(spent - 1, 0);
            }
            return false;
        };
        const auto load = [&](typename OpA::Raw &x, typename OpB::Raw &y, int k0) {
            a.load(x, Ap, g.lda, ml, k0, ke, g.nll, g.K, lane);
            if constexpr (!IMAGE) b.load(y, Bp, g.ldb, nl, k0, ke);
        };
        ask(first);
        aim(first);
        load(ra[0], rb[0], first);
        aim(first + kBK);
        load(ra[1], rb[1], first + kBK);
#pragma unroll
        for (int i = 0; i < kShare; i++) put(L[0], i);
        prepare(ra[0], rb[0], first, 0);
#pragma unroll
        for (int q = 0; q < kPairs; q++) split(q, ra[0], rb[0], fa[0], L[0], first);
        complete(ra[0], fa[0], first);
        lds_barrier();
        // One step: the products of k0's parts, beside the split of k0 + kBK's elements and the loads of k0 + 2 kBK's.
        const auto step = [&](auto parity, int k0) __attribute__((always_inline)) -> bool {
            constexpr int p = decltype(parity)::value;
            if (follow(p, ra[p])) return false;
#pragma unroll
            for (int i = 0; i < MT; i++) csum[i] += part_sum[i];
            ask(k0 + kBK);
            if (k0 + 3 * kBK > ke) aim(k0 + 2 * kBK);
            load(ra[p], rb[p], k0 + 2 * kBK);
            prepare(ra[p ^ 1], rb[p ^ 1], k0 + kBK, p ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            frag fb[2][T::kPlanes];
            const auto read = [&](int j) {
#pragma unroll
                for (int q = 0; q < T::kPlanes; q++) fb[j % 2][q] = __builtin_bit_cast(frag, L[p].u[q][0][unit[j % 2] + 16 * j]);
            };
            read(0);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int j = 0; j < NT; j++) {
                if (j + 1 < NT) read(j + 1);
#pragma unroll
                for (int q = j * kPairs / NT; q < (j + 1) * kPairs / NT; q++) split(q, ra[p ^ 1], rb[p ^ 1], fa[p ^ 1], L[p ^ 1], k0 + kBK);
                if constexpr (IMAGE)        // in the step's second half
#pragma unroll
                    for (int i = max(0, 2 * j - NT) * kShare / NT; i < max(0, 2 * j + 2 - NT) * kShare / NT; i++) put(L[p ^ 1], i);
#pragma unroll
                for (int q = 0; q < T::kProducts; q++)
#pragma unroll
                    for (int i = 0; i < MT; i++)
                        acc[i][j] = T::mma(fb[j % 2][T::kOrder[q][1]], __builtin_bit_cast(frag, fa[p][i][T::kOrder[q][0]]), acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
            complete(ra[p ^ 1], fa[p ^ 1], k0 + kBK);
            lds_barrier();
            return true;
        };
        for (int k0 = first; k0 < ke; k0 += 2 * kBK) {      // an odd number of steps: the last one's elements are zeros
            if (!step(std::integral_constant<int, 0>(), k0)) return k0;
            if (!step(std::integral_constant<int, 1>(), k0 + kBK)) return k0 + kBK;
        }
        return ke;
    };
    const int stopped = steps(S(), kb);
    if constexpr (S::kScaled)
        if (stopped < ke) {
            // the rest of k as Bf16x3, to results of the size they have
            if (b.c == 0)
#pragma unroll
                for (int t = 0; t < OpB::kUnits; t++) exponents[b.row_of(t)] = b.s[t].exponent();
            __syncthreads();
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    const v4i eb = *reinterpret_cast<const v4i *>(exponents + 16 * j + 4 * lc);
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[i][j][e] = ldexpf(acc[i][j][e], a.s[i].exponent() + eb[e]);
                }
#pragma unroll
            for (int i = 0; i < MT; i++) a.s[i].one();
#pragma unroll
            for (int t = 0; t < OpB::kUnits; t++) b.s[t].one();
            steps(Bf16x3(), stopped);
        }

    // An element that is not finite (0 times it is NaN)
    float odd = 0.f;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) odd = fmaf(acc[i][j][r], 0.f, odd);
    const bool wave_odd = __any(odd != 0.f || far);
    if (lane == 0) odd_waves[wave] = wave_odd;
    __syncthreads();
    bool odd_tile = false;
#pragma unroll
    for (int w = 0; w < WAVES; w++) odd_tile |= odd_waves[w] != 0;
    if (rarely(odd_tile)) {
        // the tile once more from the fp32 operands
#pragma unroll
        for (int i = 0; i < MT; i++) {
            a.s[i].one();
#pragma unroll
            for (int j = 0; j < NT; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int t = 0; t < OpB::kUnits; t++) b.s[t].one();
        v4f *const plain = reinterpret_cast<v4f *>(shared);
#pragma unroll 1
        for (int k0 = kb; k0 < ke; k0 += kBK) {
            aim(k0);
            load(ra[0], rb[0], k0);
            a.hand_over(ra[0], lane);
            if (ke % 4 && k0 + kBK > ke) a.cut(ra[0], k0, ke), b.cut(rb[0], k0, ke);
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int e = 0; e < 8; e++) ra[0].x[i][e] = a.element(ra[0], i, e, true, m0, k0, ke);
            b.store_plain(plain, rb[0]);
            __syncthreads();
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    const v4f y = plain[(2 * lc + h) * BN + 16 * j + lr];
#pragma unroll
                    for (int e = 0; e < 4; e++)
#pragma unroll
                        for (int i = 0; i < MT; i++)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[e], ra[0].x[i][4 * h + e], acc[i][j], 0, 0, 0);
                }
            __syncthreads();
        }
    }

    if constexpr (!AKC) {
        if (sums)      // the four k-chunks of a row
#pragma unroll
            for (int i = 0; i < MT; i++) {
                csum[i] += __shfl_xor(csum[i], 16, 64);
                csum[i] += __shfl_xor(csum[i], 32, 64);
                const int row = OpA::row_of(i, lr);
                if (lc == 0 && row < ml) g.colsum[(int64_t)range * g.M + m0 + row] = csum[i];
            }
    }
    if (b.c == 0)
#pragma unroll
        for (int t = 0; t < OpB::kUnits; t++) exponents[b.row_of(t)] = b.s[t].exponent();
    if (tid < BN) biases[tid] = g.epi.bias && g.ranges == 1 && tid < nl ? g.epi.bias[n0 + tid] : 0.f;
    __syncthreads();
    int row[MT];
    int ea[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) row[i] = OpA::row_of(i, lr), ea[i] = a.s[i].exponent();
    finish<S::kScaled, MT, NT, MODE>(g, acc, row, m0, WM, n0, lc, ea, Columns{exponents, biases}, range, id % g.tn);
}

// What two fp16 numbers leave of the small elements of rows of B that are split for a whole product: bit 8 s + e of `bits` for those at
// e of step s, `far` if one is too small even for that, and of the first kKept of those bits the values.
template <int BN>
struct Rests {
    static constexpr int kKept = 896 / BN;
    unsigned bits[2];
    int far;
    float kept[kKept][4][BN];
    static __device__ __forceinline__ int place(uint64_t all, int bit) { return __popcll(all & ((1ull << bit) - 1)); }
    __device__ __forceinline__ void clear(int tid) {
        if (tid == 0) bits[0] = bits[1] = 0, far = 0;
    }
    __device__ __forceinline__ uint64_t all() const {
        return (unsigned)__builtin_amdgcn_readfirstlane(bits[0]) | (uint64_t)(unsigned)__builtin_amdgcn_readfirstlane(bits[1]) << 32;
    }
};

// B's rows split for a whole product at once: a thread's share of THREADS threads' of BN rows x 32 KS k.  A task is a k-chunk of
// one row (KC) or of two neighbouring ones.
template <class S, bool KC, int KS, int BN, int THREADS>
struct Kept {
    static constexpr int VEC = KC ? 1 : 2, kTasks = KS * 4 * BN / VEC / THREADS;
    static_assert(kTasks >= 1, "a task per thread");
    float x[kTasks][VEC][8];

    static __device__ __forceinline__ int chunk(int task) { return KC ? task % 4 : task / (BN / 2) % 4; }
    static __device__ __forceinline__ int row(int task) { return KC ? task / 4 % BN : task % (BN / 2) * 2; }
    static __device__ __forceinline__ int step(int task) { return KC ? task / (4 * BN) : task / (2 * BN); }

    // P: the first row at the first k, `left` rows from there, K of k
    __device__ __forceinline__ void load(const float *P, int64_t ld, int left, int K, int tid) {
        const v4i rs = buffer_of(P, KC ? (int64_t)(min(left, BN) - 1) * ld + K : (int64_t)(K - 1) * ld + left);
#pragma unroll
        for (int t = 0; t < kTasks; t++) {
            const int task = tid + t * THREADS, r = row(task), k = 32 * step(task) + 4 * chunk(task);
            if constexpr (KC) {
                const unsigned at = (unsigned)(r * ld + k) * 4;
                const v4f a = llvm_raw_buffer_load_v4f32(rs, (int)(k < K ? at : kOut), 0, 0),
                          b = llvm_raw_buffer_load_v4f32(rs, (int)(k + 16 < K ? at + 64 : kOut), 0, 0);
#pragma unroll
                for (int j = 0; j < 4; j++) x[t][0][j] = a[j], x[t][0][4 + j] = b[j];
            } else {
                const unsigned at = (unsigned)(k * ld + r) * 4;
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const v2f a = llvm_raw_buffer_load_v2f32(rs, (int)(r < left ? at + (unsigned)(k_of(0, e) * ld) * 4 : kOut), 0, 0);
                    x[t][0][e] = a[0], x[t][1][e] = r + 1 < left ? a[1] : 0.f;
                }
            }
        }
    }
    // the largest magnitude of each row to `top` (LDS, zeros)
    __device__ __forceinline__ void largest(unsigned *top, int K, int tid) {
#pragma unroll
        for (int t = 0; t < kTasks; t++)
#pragma unroll
            for (int v = 0; v < VEC; v++) {
                const int task = tid + t * THREADS;
                if constexpr (KC)
#pragma unroll
                    for (int e = 0; e < 8; e++) x[t][v][e] = 32 * step(task) + k_of(chunk(task), e) < K ? x[t][v][e] : 0.f;
                atomicMax(&top[row(task) + v], __float_as_uint(abs_max8(x[t][v])));
            }
    }
    // look(task, elements, scale, split) besides
    template <class Look>
    __device__ __forceinline__ void store(Planes<S::kPlanes, BN> *L, int *exponents, const unsigned *top, int tid, Look look) const {
#pragma unroll
        for (int t = 0; t < kTasks; t++)
#pragma unroll
            for (int v = 0; v < VEC; v++) {
                const int task = tid + t * THREADS, r = row(task) + v, c = chunk(task);
                Scale s;
                s.set(__uint_as_float(top[r]), 14);
                v4u d[S::kPlanes];
#pragma unroll
                for (int j = 0; j < 4; j++) split_pair<S>(x[t][v], j, s.s, d);
                look(task, x[t][v], s.s, d);
#pragma unroll
                for (int p = 0; p < S::kPlanes; p++) L[step(task)].u[p][c][unit_of(r, c)] = d[p];
                if (step(task) == 0 && c == 0) exponents[r] = s.exponent();
            }
    }
    // a task's small elements to the bits of all
    static __device__ __forceinline__ void note_small(Rests<BN> &rests, int task, const float *y, float s, v4u *d) {
        const float least = nonzero_min8(y) * s;
        if (least < kSmall) {
            unsigned m = 0;
#pragma unroll
            for (int e = 0; e < 8; e++) m |= y[e] != 0.f && fabsf(y[e] * s) < kSmall ? 1u << e : 0u;
            atomicOr(&rests.bits[step(task) / 4], m << 8 * (step(task) % 4));
            if (least < kTiny) S::drop_tiny(d);
            if (least < kFarthest) rests.far = 1;
        }
    }
    // fp32 as it is, [step][half][chunk][row]
    __device__ __forceinline__ void store_plain(v4f (*L)[2][4][BN], int tid) const {
#pragma unroll
        for (int t = 0; t < kTasks; t++)
#pragma unroll
            for (int v = 0; v < VEC; v++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int task = tid + t * THREADS;
                    const float *const y = x[t][v] + 4 * h;
                    L[step(task)][h][chunk(task)][row(task) + v] = v4f{y[0], y[1], y[2], y[3]};
                }
    }
    // `all`: the bits of all threads' small elements
    __device__ __forceinline__ void store_rests(Rests<BN> &rests, const unsigned *top, uint64_t all, int tid) const {
#pragma unroll
        for (int t = 0; t < kTasks; t++) {
            const int task = tid + t * THREADS, first = 8 * __builtin_amdgcn_readfirstlane(step(task));
#pragma unroll 1
            for (unsigned left = (unsigned)(all >> first) & 0xff; left; left &= left - 1) {
                const int e = __builtin_ctz(left), at = Rests<BN>::place(all, first + e);
                if (at >= Rests<BN>::kKept) break;
#pragma unroll
                for (int v = 0; v < VEC; v++) {
                    Scale s;
                    s.set(__uint_as_float(top[row(task) + v]), 14);
                    rests.kept[at][chunk(task)][row(task) + v] = Half2::rest(pick(x[t][v], e) * s.s);
                }
            }
        }
    }
};

// Keeps what is computed from it in rare code from being held in registers outside
__device__ __forceinline__ int afresh(int x) {
    asm volatile("" : "+v"(x));
    return x;
}

// What is left of B's element at e of step s in row n, from memory
template <bool BKC>
__device__ __forceinline__ float rest_of(const float *Bp, int64_t ldb, int n, int nl, int k, int K, const int *exponents) {
    const float y = n < nl && k < K ? Bp[BKC ? n * ldb + k : k * ldb + n] : 0.f;
    return Half2::rest(ldexpf(y, -exponents[n]));
}

// acc += the fp32 products of a wave's rows (x: a step's elements of A) with B's rows from memory
template <bool BKC, int MT, int NT>
__device__ __forceinline__ void plain_step(v4f (&acc)[MT][NT], const float (&x)[MT][8], const float *Bp, int64_t ldb, int nl, int k0, int K,
                                           int lr, int lc) {
#pragma unroll
    for (int e = 0; e < 8; e++)
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int n = 16 * j + lr, k = k0 + k_of(lc, e);
            const float y = n < nl && k < K ? Bp[BKC ? n * ldb + k : k * ldb + n] : 0.f;
#pragma unroll
            for (int i = 0; i < MT; i++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(y, x[i][e], acc[i][j], 0, 0, 0);
        }
}

template <int MT, int NT>
__device__ __forceinline__ bool any_odd(const v4f (&acc)[MT][NT]) {      // 0 times what is not finite is NaN
    float x = 0.f;
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) x = fmaf(acc[i][j][r], 0.f, x);
    return __any(x != 0.f);
}

// Products with K up to 32 KS: a workgroup keeps 16 NT of B's rows, split, in LDS and its eight waves go over blocks of 32
// rows of A, each by itself, without barriers: one wave's results leave while others multiply.  32768 x 1024, K = 256 with bias and
// ReLU 64 us (staged 87; memory alone 35), 24576 x 2048, K = 128 with a gate 100 us (127; 87), all before the look for small elements (4 to 8 us).
template <bool BKC, int KS, int NT, int MODE>
__global__ __launch_bounds__(2 * kThreads, 2) void k_gemm_resident(GemmArgs g, int per) {
    typedef Half2 S;
    typedef S::frag frag;
    constexpr int BN = 16 * NT, MT = 2, kBlock = 16 * MT, kWaves = 8;
    typedef Direct<true, MT, false> OpA;
    __shared__ Planes<S::kPlanes, BN> L[KS];
    __shared__ unsigned top[BN];                       // the largest magnitude of each of B's rows
    __shared__ __align__(16) int exponents[2][BN];     // of the scales, zeros
    __shared__ __align__(16) float biases[BN];
    __shared__ Rests<BN> rests;
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int total = gridDim.x, xcd = blockIdx.x % 8, each = total / 8, rest = total % 8;
    const int id = xcd * each + min(xcd, rest) + blockIdx.x / 8;
    const int n0 = (id % g.tn) * BN, nl = g.N - n0, K = g.K;
    const float *const Bp = BKC ? g.B + (int64_t)n0 * g.ldb : g.B + n0;
    if (tid < BN) top[tid] = 0, exponents[1][tid] = 0, biases[tid] = g.epi.bias && tid < nl ? g.epi.bias[n0 + tid] : 0.f;
    rests.clear(tid);
    __syncthreads();
    uint64_t small_b;
    {
        Kept<S, BKC, KS, BN, 2 * kThreads> kept;
        kept.load(Bp, g.ldb, nl, K, tid);
        kept.largest(top, K, tid);
        __syncthreads();
        kept.store(L, exponents[0], top, tid, [&](int task, const float *y, float scale, v4u *d) { kept.note_small(rests, task, y, scale, d); });
        __syncthreads();
        small_b = rests.all();
        if (small_b) {
            kept.store_rests(rests, top, small_b, tid);
            __syncthreads();
        }
    }
    const bool far_b = __builtin_amdgcn_readfirstlane(rests.far);

    const int lr = lane % 16, lc = lane / 16;
    const int unit[2] = {lc * BN + unit_of(lr, lc), lc * BN + unit_of(16 + lr, lc) - 16};
    const int end = min((id / g.tn + 1) * per, (g.M + kBlock - 1) / kBlock);
    int block = id / g.tn * per + wave;
    if (block >= end) return;
    OpA a;
    a.init(lane, 0, 0, g.nll);
    const bool ragged = K < 32 * KS;
    const auto load = [&](OpA::Raw &x, int blk, int k0) {
        if (ragged) a.aim(g.lda, k0, K);
        a.load(x, g.A + (int64_t)blk * kBlock * g.lda, g.lda, blk < end ? g.M - blk * kBlock : 0, k0, K, g.nll, 0, lane);
    };
    OpA::Raw ra[2];
    v4u fa[2][MT][S::kPlanes];
    v4f acc[MT][NT];
    float change[MT];
    bool changed = false, far = false;
    bool small_a = false, zeros = false;      // zeros: A has elements that are zero, ReLU's
    // zeros beyond K, scales that the step's elements fit, and whether some are small
    const auto prepare = [&](OpA::Raw &x, int k0) __attribute__((always_inline)) {
        if (K % 4 && k0 + kBK > K) a.cut(x, k0, K);
        float m[MT];
        const bool beyond = largest_of(x.x, a.s, m) > kLargest;
        small_a = false;
        const float smallest = zeros ? smallest_nonzero_of(x.x, a.s) : smallest_of(x.x, a.s);
        if (rarely(__any(beyond || smallest < kSmall))) {
            zeros |= __any(smallest == 0.f) != 0;
            if (__any(beyond)) {
                changed = true;
#pragma unroll
                for (int i = 0; i < MT; i++) change[i] = a.s[i].fit(OpA::of_row(m[i])), far |= a.s[i].shrunk();
            }
            const float least = smallest_nonzero_of(x.x, a.s);
            small_a = __any(least < kSmall);
            far |= least < kFarthest;
        }
    };
    const auto split = [&](int q, const OpA::Raw &x, v4u (*f)[S::kPlanes]) { split_pair<S>(x.x[q % MT], q / MT, a.s[q % MT].s, f[q % MT]); };
    const auto clear = [&] {
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    };
    a.aim(g.lda, 0, 32 * KS);
    a.s[0].none(), a.s[1].none();
    load(ra[0], block, 0);
    load(ra[1], block, kBK);
    prepare(ra[0], 0);
#pragma unroll
    for (int q = 0; q < 4 * MT; q++) split(q, ra[0], fa[0]);
    for (; block < end; block += kWaves) {
        clear();
        int ea[MT];
        bool odd = far_b;
        // the products of step s, beside the split of step s + 1 and the loads of step s + 2, which may be the next block's
        const auto step = [&](auto parity, int s) __attribute__((always_inline)) {
            constexpr int p = decltype(parity)::value;
            if (rarely(changed && s > 0)) {      // results so far to the scales of step s
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int j = 0; j < NT; j++) acc[i][j] *= change[i];
            }
            changed = false;
            const unsigned b_here = (unsigned)(small_b >> 8 * s) & 0xff;
            if (rarely(small_a)) add_small(acc, ra[p].x, a.s, fa[p], L[s], unit);
            if (rarely(b_here != 0))
                add_rests(acc, ra[p].x, a.s, 0, b_here, fa[p], L[s], unit, [&](int, int e) { return b_here >> e & 1; }, [&](int j, int e) {
                    const int at = Rests<BN>::place(small_b, 8 * s + e);
                    return at < Rests<BN>::kKept ? rests.kept[at][lc][16 * j + lr]
                                                 : rest_of<BKC>(Bp, g.ldb, 16 * j + afresh(lr), nl, 32 * s + k_of(lc, e), K, exponents[0]);
                });
            load(ra[p], s + 2 < KS ? block : block + kWaves, (s + 2) % KS * kBK);
            if (s + 1 == KS) {
                odd |= far, far = false;
#pragma unroll
                for (int i = 0; i < MT; i++) ea[i] = a.s[i].exponent(), a.s[i].none();
            }
            prepare(ra[p ^ 1], (s + 1) % KS * kBK);
            __builtin_amdgcn_sched_barrier(0);
            frag fb[2][S::kPlanes];
            const auto read = [&](int j) {
#pragma unroll
                for (int q = 0; q < S::kPlanes; q++) fb[j % 2][q] = __builtin_bit_cast(frag, L[s].u[q][0][unit[j % 2] + 16 * j]);
            };
            read(0);
            if (wave < 4) __builtin_amdgcn_s_setprio(1);
            else __builtin_amdgcn_s_setprio(2);
#pragma unroll
            for (int j = 0; j < NT; j++) {
                if (j + 1 < NT) read(j + 1);
#pragma unroll
                for (int q = j * 4 * MT / NT; q < (j + 1) * 4 * MT / NT; q++) split(q, ra[p ^ 1], fa[p ^ 1]);
#pragma unroll
                for (int q = 0; q < S::kProducts; q++)
#pragma unroll
                    for (int i = 0; i < MT; i++)
                        acc[i][j] = S::mma(fb[j % 2][S::kOrder[q][1]], __builtin_bit_cast(frag, fa[p][i][S::kOrder[q][0]]), acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
            }
            __builtin_amdgcn_s_setprio(0);
        };
#pragma unroll 1
        for (int s = 0; s < KS; s += 2) {
            step(std::integral_constant<int, 0>(), s);
            step(std::integral_constant<int, 1>(), s + 1);
        }
        const int *eb = exponents[0];
        if (rarely(any_odd(acc) || __any(odd))) {
            // an element that is not finite (0 times it is NaN) or too small: the block once more from the fp32 operands
            OpA::Raw x;
            clear();
            const int r = afresh(lr);
            eb = exponents[1];
            ea[0] = ea[1] = 0;
#pragma unroll 1
            for (int k0 = 0; k0 < K; k0 += kBK) {
                load(x, block, k0);
                if (K % 4 && k0 + kBK > K) a.cut(x, k0, K);
                plain_step<BKC>(acc, x.x, Bp, g.ldb, nl, k0, K, r, lc);
            }
        }
        int row[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) row[i] = OpA::row_of(i, lr);
        finish<true, MT, NT, MODE>(g, acc, row, block * kBlock, kBlock, n0, lc, ea, Columns{eb, biases}, 0, id % g.tn);
    }
}

// Small products, 64 x 64 tiles with up to 32 KS k each: everything is asked for at once and split as it arrives, three barriers in
// all.  Bound by latency, one trip to memory and a chain of 12 KS matrix instructions: 300 x 256, K = 256 7.0 us (step by step
// 8.5; 2 are an empty kernel's), 300 x 128, K = 128 4.6 (6.3), x^T y of 1000 rows, 1024 x 256 11.6 with the ranges' sum (15.8).
template <bool AKC, bool BKC, int KS, int MODE>
__global__ __launch_bounds__(kThreads, 2) void k_gemm_once(GemmArgs g) {
    typedef WideHalf2 S;
    constexpr int NT = 4, BN = 16 * NT;
    typedef Direct<AKC, 1, false> OpA;
    __shared__ Planes<S::kPlanes, BN> L[KS];
    __shared__ unsigned top[BN];
    __shared__ __align__(16) int exponents[2][BN];
    __shared__ __align__(16) float biases[BN];
    __shared__ int odd;
    const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), lr = lane % 16, lc = lane / 16;
    const int total = gridDim.x, xcd = blockIdx.x % 8, each = total / 8, rest = total % 8;
    const int tile = xcd * each + min(xcd, rest) + blockIdx.x / 8, range = tile / (g.tm * g.tn), id = tile % (g.tm * g.tn);
    const int m0 = id / g.tn * 64 + wave * 16, n0 = id % g.tn * BN, ml = g.M - m0, nl = g.N - n0;
    const int kb = range * g.ks, K = min(g.K - kb, g.ks);
    const float *const Ap = AKC ? g.A + (int64_t)m0 * g.lda + kb : g.A + m0 + kb * g.lda;
    const float *const Bp = BKC ? g.B + (int64_t)n0 * g.ldb + kb : g.B + n0 + kb * g.ldb;
    if (tid < BN) top[tid] = 0, exponents[1][tid] = 0, biases[tid] = g.epi.bias && g.ranges == 1 && tid < nl ? g.epi.bias[n0 + tid] : 0.f;
    if (tid == 0) odd = 0;
    Kept<S, BKC, KS, BN, kThreads> kept;
    OpA a;
    typename OpA::Raw x[KS];
    kept.load(Bp, g.ldb, nl, K, tid);
    a.init(lane, m0, g.M, g.nll);
    const auto load = [&](typename OpA::Raw &y, int k0) {
        a.aim(g.lda, k0, K);
        a.load(y, Ap, g.lda, ml, k0, K, g.nll, 0, lane);
    };
#pragma unroll
    for (int s = 0; s < KS; s++) load(x[s], 32 * s);
    lds_barrier();
    kept.largest(top, K, tid);
    lds_barrier();
    kept.store(L, exponents[0], top, tid, [&](int, const float *y, float scale, v4u *) {
        if (nonzero_min8(y) * scale < S::kLeast) odd = 1;
    });
    float m = 0.f, csum = 0.f;
#pragma unroll
    for (int s = 0; s < KS; s++) {
        if (K % 4 && 32 * s + 32 > K) a.cut(x[s], 32 * s, K);
        m = fmaxf(m, abs_max8(x[s].x[0]));
    }
    a.s[0].set(OpA::of_row(m), 14);
    if constexpr (!AKC) {
        if (g.colsum && n0 == 0)
#pragma unroll
            for (int s = 0; s < KS; s++)
#pragma unroll
                for (int e = 0; e < 8; e++) csum += x[s].x[0][e];
    }
    lds_barrier();
    v4f acc[1][NT], low[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) acc[0][j] = low[j] = v4f{0.f, 0.f, 0.f, 0.f};
    const int unit[2] = {lc * BN + unit_of(lr, lc), lc * BN + unit_of(16 + lr, lc) - 16};
#pragma unroll
    for (int s = 0; s < KS; s++) {
        v4u f[S::kPlanes];
#pragma unroll
        for (int q = 0; q < 4; q++) split_pair<S>(x[s].x[0], q, a.s[0].s, f);
#pragma unroll
        for (int q = 0; q < S::kProducts; q++)
#pragma unroll
            for (int j = 0; j < NT; j++) {
                v4f &to = S::kOrder[q][0] + S::kOrder[q][1] ? low[j] : acc[0][j];
                to = S::mma(__builtin_bit_cast(S::frag, L[s].u[S::kOrder[q][1]][0][unit[j % 2] + 16 * j]),
                            __builtin_bit_cast(S::frag, f[S::kOrder[q][0]]), to);
            }
    }
#pragma unroll
    for (int j = 0; j < NT; j++) acc[0][j] += low[j] * S::kRest;
    bool far = any_odd(acc);
#pragma unroll
    for (int s = 0; s < KS; s++) far |= smallest_nonzero_of(x[s].x, a.s) < S::kLeast;
    if (far) odd = 1;
    const int *eb = exponents[0];
    int ea[1] = {a.s[0].exponent()}, row[1] = {OpA::row_of(0, lr)};
    __syncthreads();
    if (odd) {
        // the tile once more in fp32, B through LDS: 15.5 us for 2000 rows of very different sizes, x^T y, 256 x 128 (11.3 without; B from memory 37.6)
        eb = exponents[1], ea[0] = 0;
#pragma unroll
        for (int j = 0; j < NT; j++) acc[0][j] = v4f{0.f, 0.f, 0.f, 0.f};
        v4f(*const plain)[2][4][BN] = reinterpret_cast<v4f(*)[2][4][BN]>(L);
        kept.store_plain(plain, tid);
        __syncthreads();
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int j = 0; j < NT; j++) {
                    const v4f y = plain[s][h][lc][16 * j + lr];
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[0][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[e], x[s].x[0][4 * h + e], acc[0][j], 0, 0, 0);
                }
    }
    if constexpr (!AKC)
        if (g.colsum && n0 == 0) {
            csum = csum + __shfl_xor(csum, 16, 64);
            csum += __shfl_xor(csum, 32, 64);
            if (lc == 0 && lr < ml) g.colsum[(int64_t)range * g.M + m0 + lr] = csum;
        }
    finish<true, 1, NT, MODE>(g, acc, row, m0, 16, n0, lc, ea, Columns{eb, biases}, range, id % g.tn);
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

template <class S, bool AKC, bool BKC, int MODE>
void launch_staged(const GemmArgs &g, const Plan &p, hipStream_t s) {
    const dim3 grid((unsigned)(p.tm * p.tn * p.ranges));
    if (p.bm == 64) hipLaunchKernelGGL((k_gemm<S, AKC, BKC, 1, 4, MODE>), grid, dim3(kThreads), 0, s, g);
    else if (p.bn == 64) hipLaunchKernelGGL((k_gemm<S, AKC, BKC, 2, 4, MODE>), grid, dim3(kThreads), 0, s, g);
    else hipLaunchKernelGGL((k_gemm<S, AKC, BKC, 2, 8, MODE>), grid, dim3(kThreads), 0, s, g);
}

// The loss gradient's products stay with Bf16x3: a word's probabilities over the tokens, or a token's over the words, are
// held to their own size, however far below the largest.
template <bool AKC, bool BKC, int MODE>
void launch(GemmArgs g, const Plan &p, hipStream_t s) {
    g.ks = p.ks, g.tm = p.tm, g.tn = p.tn, g.ranges = p.ranges;
    if constexpr (MODE == kGrad) {
        if (g.image) {
            const dim3 steps((unsigned)((g.K + kBK - 1) / kBK), (unsigned)g.tn), grid((unsigned)(g.tm * g.tn * g.ranges));
            if (p.bn == 256) {
                hipLaunchKernelGGL(k_image<256>, steps, dim3(512), 0, s, g.B, g.ldb, g.N, g.K, g.image);
                hipLaunchKernelGGL((k_gemm<Bf16x3, AKC, BKC, 1, 16, MODE, 8, true>), grid, dim3(512), 0, s, g);
            } else {
                hipLaunchKernelGGL(k_image<128>, steps, dim3(256), 0, s, g.B, g.ldb, g.N, g.K, g.image);
                hipLaunchKernelGGL((k_gemm<Bf16x3, AKC, BKC, 2, 8, MODE, 4, true>), grid, dim3(256), 0, s, g);
            }
        } else if (p.bn == 256)
            hipLaunchKernelGGL((k_gemm<Bf16x3, AKC, BKC, 1, 16, MODE, 8>), dim3((unsigned)(g.tm * g.tn * g.ranges)), dim3(512), 0, s, g);
        else
            launch_staged<Bf16x3, AKC, BKC, MODE>(g, p, s);
    }
    else if (g.K < kHalfK) launch_staged<Bf16x3, AKC, BKC, MODE>(g, p, s);
    else {
        if constexpr (AKC) {
            if (p.steps) {
                g.tn = (g.N + 127) / 128;
                const dim3 grid((unsigned)(g.tn * p.groups)), block(2 * kThreads);
                if (p.steps == 4) hipLaunchKernelGGL((k_gemm_resident<BKC, 4, 8, MODE>), grid, block, 0, s, g, p.per);
                else hipLaunchKernelGGL((k_gemm_resident<BKC, 8, 8, MODE>), grid, block, 0, s, g, p.per);
                return;
            }
        }
        if (p.once) {
            const dim3 grid((unsigned)(p.tm * p.tn * p.ranges));
            if (p.ks <= 128) hipLaunchKernelGGL((k_gemm_once<AKC, BKC, 4, MODE>), grid, dim3(kThreads), 0, s, g);
            else hipLaunchKernelGGL((k_gemm_once<AKC, BKC, 8, MODE>), grid, dim3(kThreads), 0, s, g);
            return;
        }
        launch_staged<Half2, AKC, BKC, MODE>(g, p, s);
    }
}

bool aligned(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace

int matmul(int layout, const float *A, int64_t lda, const float *B, int64_t ldb, float *C, int64_t ldc, int M, int N,
           int K, const fwp_mm_epilogue &epi, float *workspace, const NllView *nll, hipStream_t s) {
    GemmArgs g{};
    g.A = A, g.B = B, g.lda = lda, g.ldb = ldb, g.M = M, g.N = N, g.K = K, g.epi = epi;
    if (nll) g.nll = NllArgs{nll->lse, nll->stats, nll->gloss, nll->target, nll->vocab};
    const Scratch scratch = scratch_of(M, N, K, workspace && ldc == N && aligned(C) && aligned(workspace), nll != nullptr);
    const Plan &p = scratch.plan;
    const bool cut = p.ranges > 1;
    if (scratch.image) g.image = reinterpret_cast<v4u *>(workspace + scratch.parts);
    g.C = cut ? workspace : C;
    g.ldc = cut ? N : ldc;
    g.part = part_of(M, N);
    g.vec = g.ldc % 4 == 0 && N % 4 == 0 && aligned(g.C) && aligned(epi.residual) && aligned(epi.gate);
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
    const Plan p = plan_of(rows, vocab, dim, false, false);
    const int tn = p.steps ? (vocab + 127) / 128 : p.tn;
    g.part_max = workspace;
    g.part_sum = workspace + (int64_t)tn * rows;
    g.hit = logits ? nullptr : g.part_sum + (int64_t)tn * rows;
    g.vec = vocab % 4 == 0 && aligned(logits);
    launch<true, true, kLse>(g, p, s);
    hipLaunchKernelGGL(k_nll, dim3((rows + 63) / 64), dim3(kThreads), 0, s, g.part_max, g.part_sum, g.hit, logits, target, loss,
                       lse, stats, rows, vocab, tn);
    return (int)hipGetLastError();
}

}  // namespace fwp
