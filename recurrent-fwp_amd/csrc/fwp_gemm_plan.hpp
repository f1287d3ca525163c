// Which kernel a matrix product takes, in which tiles, and how much of the caller's workspace it uses: of sizes and alignment alone, without a device.
#pragma once
#include <algorithm>
#include <cstdint>

namespace fwp {

constexpr int kBK = 32;               // k per LDS tile
constexpr int kImagePlanes = 3;       // numbers of 16 bits to an element of the split operand's image

// Which kernel: the one with B's rows kept in LDS (`steps` of k, 4 or 8; `per` blocks of 32 rows to a workgroup, `groups` of
// them), the one that asks for everything at once (`once`, tiles of 64 x 64), or the staged one with tiles of bm x bn; k in `ranges` of ks.
struct Plan {
    int steps, per, groups;
    bool once;
    int bm, bn, tm, tn, ranges, ks;
};

// Kept rows of B, from 128 to 256 k and where workgroups of 256 rows x 128 columns are enough for most CUs: 32768 x 1024,
// K = 256 64 us (staged 87, both with bias and ReLU), 24576 x 2048, K = 128 with a gate 100 us (staged 127), 8192 x 776, K = 256
// (224 workgroups) 19 us (22); 16384 x 256, K = 256 (128 workgroups) 19 us (16), 8192 x 392, K = 128 (128) 13 us (11).
constexpr int kResidentTiles = 200;
// Half2's error is the smaller one from here on; below, Bf16x3's (K = 64: 1.08e-7 and 1.06e-7, K = 32: 8.8e-8 and 6.3e-8).
constexpr int kHalfK = 128;

// (These times and those below are without the look for small elements, which takes a tenth on either side.)
// Staged: 128 x 128 tiles where, with k cut into ranges, they are three for two CUs; else 128 x 64 if those are; else 64 x 64.
// 32768 x 256, K = 1024 (512 tiles) 60 us, 77, 80; 16384 x 256, K = 1024 (256 tiles) 47, 41, 48 us; 2381 x 1024, K = 256
// (152, 304, 608 tiles) 16.2, 15.9, 14.3 us; 300 x 256, K = 256 13.9, 10.3, 8.6 us.  Those of 64 x 64 all at once where a tile's k
// is at most 256 or can be cut into ranges that are, and that makes no more than two workgroups for a CU: 300 x 256, K = 256
// 7.0 us, 1000 x 256, K = 1024 (256 workgroups) 11.9 us staged 13.2, 2381 x 256, K = 1024 (608) 20.8 us, staged 19.1.
// The partial results of a range cost a pass over M x N each way, so a range is no shorter than 256 of k; all at once, 129.
// The loss's gradients (`grad`): 128 x 256 tiles of eight waves, which form an element once for twice the columns, where those divide over the
// chip as well as 128 x 128 ones, one of them to a CU or two of the others, the latter 1.12 times as long.  dX and dW, tokens = words = 32768: 256 columns
// 3.09 and 3.36 ms (128-column tiles 3.45, 3.85; these and the next before kImage's), 288 (512 tiles, two turns) 5.85 and 6.61 (768 tiles, one and a half: 5.10, 5.94); 8192, in two
// ranges: 288 columns 0.37 and 0.43 ms (0.38, 0.46); 640 (192 tiles) 0.69 and 0.83 (128 x 64 tiles 0.81, 1.05).
inline Plan plan_of(int M, int N, int K, bool may_cut, bool grad) {
    Plan p{};
    const auto tiles = [&](int bm, int bn) { return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
    const auto ranges = [&](int64_t tiles) { return may_cut ? std::max<int64_t>(1, std::min<int64_t>(512 / tiles, K / 256)) : 1; };
    const int blocks = (M + 31) / 32;
    if (!grad && K >= kHalfK && K <= 256 && tiles(256, 128) >= kResidentTiles) {
        p.steps = K <= 128 ? 4 : 8;
        // the most even division of the blocks over 256 CUs, a workgroup's start (its rows of B) as long as a wave's block: of those that
        // take as many turns of 256 workgroups the one with most, and of those whose waves have as many blocks that with fewest
        int64_t best = INT64_MAX;
        const int tn = (N + 127) / 128, most = std::min((blocks + 7) / 8, std::max(1, 1024 / tn));
        for (int turns = (tn + 255) / 256, n = 0; n < most; turns++) {
            n = std::min(most, 256 * turns / tn);
            const int each = ((blocks + n - 1) / n + 7) / 8, least = (blocks + 8 * each - 1) / (8 * each);
            const int64_t cost = (int64_t)turns * (each + 1);
            if (cost < best) best = cost, p.per = (blocks + least - 1) / least, p.groups = (blocks + p.per - 1) / p.per;
        }
    }
    p.bm = p.bn = 128;
    const int64_t wide = tiles(128, 128), turns = tiles(128, 256) * ranges(wide);
    if (wide * ranges(wide) < 384 && !(grad && N > 128 && turns >= 160)) {
        p.bn = 64;
        if (tiles(128, 64) < 384) p.bm = 64;
    }
    if (grad && N > 128 && p.bn == 128 && (turns + 255) / 256 <= 1.12 * std::max(1.0, wide * ranges(wide) / 512.0)) p.bn = 256;
    p.tm = (M + p.bm - 1) / p.bm;
    p.tn = (N + p.bn - 1) / p.bn;
    int64_t n = ranges(p.bn == 256 ? wide : tiles(p.bm, p.bn));
    if (!grad && p.bm == 64 && K >= kHalfK) {
        const int64_t parts = (K + 255) / 256;
        if (parts == 1 || (may_cut && parts * tiles(64, 64) <= 512)) p.once = true, n = parts;
    }
    const int whole = p.once ? kBK : 2 * kBK;
    p.ks = (int)((K + n - 1) / n + whole - 1) / whole * whole;
    p.ranges = (K + p.ks - 1) / p.ks;
    return p;
}

// a partial result, in whole 16-byte groups
inline int64_t part_of(int M, int N) { return ((int64_t)M * N + 3) / 4 * 4; }

// The loss's gradients split their second operand (the weights, the tokens) once, for all rows of tiles, where these are many and k is long: each workgroup
// did it again for its 128 rows, a third of its vector instructions, which bound them as much as the products do (each busy 45 % of the time).
// Words = tokens = 32768, 256 columns: dX 2.98 -> 2.60 ms, dW 3.19 -> 3.06 ms; 32768 words, 24576 tokens, 128 columns 1.58 -> 1.32 and
// 1.44 -> 1.25 ms; 4100 tokens, 5001 words, 256 columns 82 -> 75 and 84 -> 83 us; 3000 of both 45 -> 45 and 47 -> 50 us; 1024
// tokens, 32768 words dX 107 -> 112 us; 32768 tokens, 1024 words dW 114 -> 128 us.  With k of 1024 dX would still gain (100 -> 94 us), dW not.
constexpr int kImage = 4096;

// floats of the partial results and, behind them, of B's image
inline int64_t parts_of(const Plan &p, int M, int N) { return p.ranges > 1 ? (p.ranges * (part_of(M, N) + M) + 3) / 4 * 4 : 0; }
inline int64_t image_of(const Plan &p, int M, int K) {
    return p.bm == 128 && p.bn >= 128 && std::min(M, K) >= kImage ? (int64_t)p.tn * ((K + kBK - 1) / kBK) * (kImagePlanes * kBK / 2) * p.bn : 0;
}

// What a call does and what it uses of its workspace.  may_cut: there is a workspace, and it and the result can be taken 16 bytes at a time.  Without, the plan
// is another one, with another image, which the workspace was not measured for: no image either.
struct Scratch {
    Plan plan;
    int64_t parts, image;
};
inline Scratch scratch_of(int M, int N, int K, bool may_cut, bool grad) {
    const Plan p = plan_of(M, N, K, may_cut, grad);
    return {p, parts_of(p, M, N), grad && may_cut ? image_of(p, M, K) : 0};
}

// what a product uses (no image: 4096 x 1024 over 32768 tokens 34 MB, with the room for one 235)
inline int64_t product_workspace(int M, int N, int K) { return scratch_of(M, N, K, true, false).parts; }

// enough for a product and for a loss's gradient
inline int64_t matmul_workspace(int M, int N, int K) {
    const Scratch grad = scratch_of(M, N, K, true, true);
    return std::max(product_workspace(M, N, K), grad.parts + grad.image);
}

}  // namespace fwp
