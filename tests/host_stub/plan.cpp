// csrc/fwp_gemm_plan.hpp for the host: what the loss's gradients use of a workspace against what it was said to take.
#include "../../recurrent-fwp_amd/csrc/fwp_gemm_plan.hpp"

using namespace fwp;

extern "C" {

int64_t plan_workspace(int rows, int vocab, int dim) { return std::max(matmul_workspace(rows, dim, vocab), matmul_workspace(vocab, dim, rows)); }

// the larger use of the two gradients' products; aligned: their results lie on 16-byte boundaries
int64_t plan_used(int rows, int vocab, int dim, int aligned) {
    const Scratch dx = scratch_of(rows, dim, vocab, aligned, true), dw = scratch_of(vocab, dim, rows, aligned, true);
    return std::max(dx.parts + dx.image, dw.parts + dw.image);
}

// a product's, with and without a result on such a boundary
int64_t plan_product_used(int M, int N, int K, int aligned) {
    const Scratch s = scratch_of(M, N, K, aligned, false);
    return s.parts + s.image;
}

int64_t plan_product_workspace(int M, int N, int K) { return product_workspace(M, N, K); }
}
