"""The language model's matrix products, negative log-likelihood and LayerNorm kernels through the C ABI, against
float64.  Tolerance of a product: every one of the up to six roundings per 32 terms, and the split of an operand into
three bf16 numbers (K < 128), is at most 2^-24 of the sum of the terms' magnitudes.  Two fp16 numbers (K >= 128, where the bound is
36 times that or more) hold an element to 2^-23 of itself, a small one of its row to 2^-19 or apart."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -24
NT, NN, TN = 0, 1, 2


def bound(K, mag):
    return (6 * (K // 32 + 2)) * EPS * mag + 1e-30


def randn(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).cuda()


def matmul(L, layout, A, B, cut=True, **epi):
    K = A.shape[0] if layout == TN else A.shape[1]
    M = A.shape[1] if layout == TN else A.shape[0]
    N = B.shape[0] if layout == NT else B.shape[1]
    C = torch.full((M, N), float("nan"), device="cuda")
    e = L.Epilogue(*(epi[n].data_ptr() if n in epi else None for n in ("bias", "residual", "gate", "colsum")),
                   int(epi.get("relu", 0)))
    work = torch.empty(max(1, L.lib().fwp_matmul_workspace(M, N, K)), device="cuda") if cut else None
    rc = L.lib().fwp_matmul(layout, A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), C.data_ptr(), N, M, N, K,
                            ctypes.byref(e), work.data_ptr() if cut else None, L.stream_of(A))
    assert rc == 0, L.strerror(rc)
    return C


# the edges of the 64 and 128 tiles and of the 32-wide steps of k; few tiles and a long k (cut into ranges)
SHAPES = [(1, 1, 1), (3, 5, 7), (64, 64, 32), (65, 63, 33), (128, 128, 256), (130, 776, 256), (257, 36, 1000),
          (2048, 2049, 40), (16, 256, 4096), (776, 256, 3001), (200, 260, 8192)]


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("layout", [NT, NN, TN])
def test_products(fwp, layout, M, N, K):
    A = randn(*((K, M) if layout == TN else (M, K)), seed=1)
    B = randn(*((N, K) if layout == NT else (K, N)), seed=2)
    a, b = A.double(), B.double()
    a, b = (a.t() if layout == TN else a), (b.t() if layout == NT else b)
    want, mag = a @ b, a.abs() @ b.abs()
    for cut in (True, False):
        got = matmul(fwp._lib, layout, A, B, cut)
        assert bool(((got.double() - want).abs() <= bound(K, mag)).all())
    # operands of any size: fp32's exponents, no scaling
    got = matmul(fwp._lib, layout, A * 1e-30, B * 1e25)
    assert bool(((got.double() / 1e-5 - want).abs() <= 2 * bound(K, mag)).all())


@pytest.mark.parametrize("M,N,K", [(130, 776, 256), (64, 256, 4096)])      # one range of k, several
def test_epilogues_and_column_sums(fwp, M, N, K):
    A, B = randn(M, K, seed=1), randn(N, K, seed=2)
    bias, residual, gate = randn(N, seed=3) * 30, randn(M, N, seed=4) * 30, randn(M, N, seed=5)
    raw, mag = A.double() @ B.double().t(), A.double().abs() @ B.double().abs().t()
    got = matmul(fwp._lib, NT, A, B, bias=bias, relu=1, residual=residual, gate=gate)
    want = torch.where(gate > 0, torch.relu(raw + bias.double()) + residual.double(), 0.0)
    assert bool(((got.double() - want).abs() <= bound(K, mag + 400)).all())
    # TN: the columns of A summed over k
    G, X = randn(K, M, seed=6), randn(K, N, seed=7)
    colsum = torch.full((M,), float("nan"), device="cuda")
    got = matmul(fwp._lib, TN, G, X, colsum=colsum)
    assert bool(((got.double() - G.double().t() @ X.double()).abs() <= bound(K, G.double().abs().t() @ X.double().abs())).all())
    assert bool(((colsum.double() - G.double().sum(0)).abs() <= K * EPS * G.double().abs().sum(0)).all())


@pytest.mark.parametrize("rows,vocab,dim", [(1, 5, 4), (70, 211, 64), (64, 64, 36), (300, 4099, 128), (520, 33000, 256), (6500, 6600, 132),
                                            (70, 33000, 288), (600, 8200, 640)])
def test_negative_log_likelihood(fwp, rows, vocab, dim):
    L = fwp._lib
    x, W, b = randn(rows, dim, seed=1), randn(vocab, dim, seed=2) * 0.3, randn(vocab, seed=3)
    target = torch.randint(0, vocab, (rows,), generator=torch.Generator().manual_seed(4)).cuda()
    target[rows // 2] = -100 if rows > 1 else target[0]          # ignored
    gloss = randn(rows, seed=5)
    logits, loss, lse = (torch.full(s, float("nan"), device="cuda") for s in ((rows, vocab), (rows,), (rows,)))
    work = torch.empty(L.lib().fwp_nll_workspace(rows, vocab), device="cuda")
    ptrs = [t.data_ptr() for t in (x, W, b, target)]
    assert L.lib().fwp_nll_fwd(*ptrs, logits.data_ptr(), loss.data_ptr(), lse.data_ptr(), work.data_ptr(), rows, vocab,
                               dim, L.stream_of(x)) == 0
    only = torch.empty_like(loss)
    assert L.lib().fwp_nll_fwd(*ptrs, None, only.data_ptr(), None, work.data_ptr(), rows, vocab, dim, L.stream_of(x)) == 0
    assert torch.equal(only, loss)
    xd, Wd, bd = (t.double().requires_grad_() for t in (x, W, b))
    want = torch.nn.functional.cross_entropy(xd @ Wd.t() + bd, target, reduction="none")
    # the logits' rounding, and the hardware exponential's and logarithm's (2^-21 of the largest)
    err = bound(dim, x.double().abs() @ W.double().abs().t() + bd.abs()).max() + 2.0 ** -20
    assert float((loss.double() - want.detach()).abs().max()) <= float(err)
    gx, gW, gb = torch.full_like(x, float("nan")), torch.full_like(W, float("nan")), torch.full_like(b, float("nan"))
    n = max(L.lib().fwp_matmul_workspace(rows, dim, vocab), L.lib().fwp_matmul_workspace(vocab, dim, rows))
    work = torch.empty(n, device="cuda")
    assert L.lib().fwp_nll_bwd(x.data_ptr(), W.data_ptr(), logits.data_ptr(), lse.data_ptr(), target.data_ptr(),
                               gloss.data_ptr(), gx.data_ptr(), gW.data_ptr(), gb.data_ptr(), work.data_ptr(), rows, vocab,
                               dim, L.stream_of(x)) == 0
    wants = torch.autograd.grad(want, (xd, Wd, bd), gloss.double())
    # a probability is off by its logit's error, relatively: 2 err of the gradient's magnitude
    p = torch.softmax((xd @ Wd.t() + bd).detach(), -1)
    d = (p + torch.nn.functional.one_hot(target.clamp_min(0), vocab)) * gloss.double().abs()[:, None]
    mags = (d @ Wd.detach().abs(), d.t() @ xd.detach().abs(), d.sum(0))
    for name, got, w, mag in zip("xWb", (gx, gW, gb), wants, mags):
        assert bool(((got.double() - w).abs() <= (2 * float(err) + bound(max(rows, vocab), 1.0)) * mag + 1e-12).all()), name


def loss_and_gradients(L, x, W, b, target, gloss):
    """The loss with and without a graph's buffers (they agree), and the gradients of x, W and b."""
    rows, vocab, dim = x.shape[0], *W.shape
    logits, loss, stats = (torch.full(s, float("nan"), device="cuda") for s in ((rows, vocab), (rows,), (rows, 2)))
    work = torch.empty(L.lib().fwp_nll_workspace(rows, vocab), device="cuda")
    ptrs = [t.data_ptr() for t in (x, W, b, target)]
    assert L.lib().fwp_nll_stats_fwd(*ptrs, logits.data_ptr(), loss.data_ptr(), stats.data_ptr(), work.data_ptr(), rows, vocab,
                                     dim, L.stream_of(x)) == 0
    only = torch.empty_like(loss)
    assert L.lib().fwp_nll_fwd(*ptrs, None, only.data_ptr(), None, work.data_ptr(), rows, vocab, dim, L.stream_of(x)) == 0
    assert torch.equal(only.nan_to_num(-1.0), loss.nan_to_num(-1.0))
    gx, gW, gb = torch.full_like(x, float("nan")), torch.full_like(W, float("nan")), torch.full_like(b, float("nan"))
    n = max(L.lib().fwp_matmul_workspace(rows, dim, vocab), L.lib().fwp_matmul_workspace(vocab, dim, rows))
    work = torch.empty(max(1, n), device="cuda")
    assert L.lib().fwp_nll_stats_bwd(x.data_ptr(), W.data_ptr(), logits.data_ptr(), stats.data_ptr(), target.data_ptr(),
                                     gloss.data_ptr(), gx.data_ptr(), gW.data_ptr(), gb.data_ptr(), work.data_ptr(), rows, vocab,
                                     dim, L.stream_of(x)) == 0
    return loss, gx, gW, gb


def check_loss(L, x, W, b, target):
    gloss = randn(x.shape[0], seed=5)
    got = loss_and_gradients(L, x, W, b, target, gloss)
    xd, Wd, bd = (t.double().requires_grad_() for t in (x, W, b))
    want = torch.nn.functional.cross_entropy(xd @ Wd.t() + bd, target, reduction="none")
    wants = (want.detach(), *torch.autograd.grad(want, (xd, Wd, bd), gloss.double()))
    for name, g, w in zip(("loss", "x", "W", "bias"), got, wants):
        # K = 64 products' roundings of logits of up to about 30, as errors of probabilities, over up to 64 tokens
        assert float((g.double() - w).abs().max()) <= 2e-5 * (1 + float(w.abs().max())), name


# 64-wide tiles (few tokens) and 128-wide ones; masked: the first tile, one in the middle, all but a few words
@pytest.mark.parametrize("rows,vocab", [(70, 1000), (2048, 2200)])
@pytest.mark.parametrize("masked", [(0, 128), (640, 768), (130, 520), (0, 960)])
def test_loss_of_a_vocabulary_masked_in_part(fwp, rows, vocab, masked):
    """A bias of -infinity takes words out: whole tiles of logits are -infinity."""
    x, W, b = randn(rows, 64, seed=1), randn(vocab, 64, seed=2) * 0.3, randn(vocab, seed=3)
    b[masked[0]:masked[1]] = -float("inf")
    free = torch.nonzero(b.isfinite())[:, 0]
    target = free[torch.randint(0, len(free), (rows,), generator=torch.Generator().manual_seed(4)).cuda()]
    check_loss(fwp._lib, x, W, b, target)


@pytest.mark.parametrize("rows", [1, 31, 33, 70])
def test_loss_gradients_of_far_negative_logits(fwp, rows):
    """A softmax does not mind a shift: logits around -100, token counts that do not fill the products' steps."""
    x, W, b = randn(rows, 64, seed=1) * 0.1, randn(300, 64, seed=2) * 0.3, torch.full((300,), -100.0, device="cuda")
    target = torch.randint(0, 300, (rows,), generator=torch.Generator().manual_seed(4)).cuda()
    check_loss(fwp._lib, x, W, b, target)


@pytest.mark.parametrize("top", [1.0, 20.0, 200.0])
@pytest.mark.parametrize("vocab", [130, 1000])
def test_loss_of_confident_tokens(fwp, vocab, top):
    """Exact logits (x is the identity, W has few bits), the target's far above the others: losses down to 1e-6."""
    rows = 64
    g = torch.Generator().manual_seed(1)
    W = (torch.randint(-8, 9, (vocab, rows), generator=g) / 4.0 + (top - 18 * torch.rand(rows, generator=g)).round()).cuda()
    target = torch.randint(0, vocab, (rows,), generator=g).cuda()
    W[target, torch.arange(rows, device="cuda")] = top
    gloss = randn(rows, seed=5)
    loss, gx, gW, gb = loss_and_gradients(fwp._lib, torch.eye(rows, device="cuda"), W, torch.zeros(vocab, device="cuda"), target, gloss)
    logits = W.t().double()
    want = torch.nn.functional.cross_entropy(logits, target, reduction="none")
    # a sum of about 20 roundings, at most, and its logarithm's; the difference of two logits is exact
    assert bool(((loss.double() - want).abs() <= 32 * EPS * (1 + want)).all())
    p = torch.softmax(logits, -1)
    d = (p - torch.nn.functional.one_hot(target, vocab)) * gloss.double()[:, None]
    # the exponential's argument is rounded twice on its way to a power of two; the target's p - 1 has its roundings at 1
    hit = torch.nn.functional.one_hot(target, vocab)
    tol = EPS * gloss.double().abs()[:, None] * (p * (32 + 2 * (logits.amax(-1, keepdim=True) - logits)) + 4 * hit)
    assert bool(((gW.t().double() - d).abs() <= tol + 1e-12).all())


@pytest.mark.parametrize("vocab", [130, 1000])
def test_probabilities_far_below_the_largest(fwp, vocab):
    """Exact logits down to 80 below the largest: the exponential's own error is a few roundings there too."""
    rows, g = 64, torch.Generator().manual_seed(1)
    W = (-torch.randint(0, 321, (vocab, rows), generator=g) / 4.0).cuda()
    target = torch.randint(0, vocab, (rows,), generator=g).cuda()
    gloss = randn(rows, seed=5)
    loss, gx, gW, gb = loss_and_gradients(fwp._lib, torch.eye(rows, device="cuda"), W, torch.zeros(vocab, device="cuda"), target, gloss)
    logits = W.t().double()
    want = torch.nn.functional.cross_entropy(logits, target, reduction="none")
    assert bool(((loss.double() - want).abs() <= 16 * EPS * (1 + want)).all())
    p, hit = torch.softmax(logits, -1), torch.nn.functional.one_hot(target, vocab)
    # the exponential 3 roundings, the sum and its inverse up to 16, two products; the target's p - 1 has its own at 1
    # and an operand of the product loses what of its three parts is below the smallest normal number, 2^-126
    tol = EPS * gloss.double().abs()[:, None] * (24 * p + 4 * hit) + 2.0 ** -125
    assert bool(((gW.t().double() - (p - hit) * gloss.double()[:, None]).abs() <= tol).all())


def spread(t, by=0, first=0):
    """The same values with rows `by` floats further apart, the first `first` floats into the storage; NaN around them."""
    R, C = t.shape
    buf = torch.full((R * (C + by) + first,), float("nan"), device="cuda")
    out = buf[first:].view(R, C + by)[:, :C]
    out.copy_(t)
    return out


# results whose rows are no whole 16-byte groups: k in several ranges, in one; wide tiles and small ones
@pytest.mark.parametrize("M,N,K,cut", [(66, 201, 2400, True), (256, 1001, 700, True), (5, 3, 9000, True), (130, 775, 256, False),
                                       (2100, 2101, 64, False)])
@pytest.mark.parametrize("layout", [NT, NN, TN])
def test_ragged_results_spread_and_unaligned_operands(fwp, layout, M, N, K, cut):
    assert (fwp._lib.lib().fwp_matmul_workspace(M, N, K) > 0) == cut
    A = randn(*((K, M) if layout == TN else (M, K)), seed=1)
    B = randn(*((N, K) if layout == NT else (K, N)), seed=2)
    bias, residual, gate = randn(N, seed=3) * 30, randn(M, N, seed=4) * 30, randn(M, N, seed=5)
    a, b = A.double(), B.double()
    a, b = (a.t() if layout == TN else a), (b.t() if layout == NT else b)
    raw, mag = a @ b, a.abs() @ b.abs()
    want = torch.where(gate > 0, torch.relu(raw + bias.double()) + residual.double(), 0.0)
    for by, first in ((0, 0), (0, 1), (3, 2), (8, 4)):
        x, y = spread(A, by, first), spread(B, by, first)
        if layout == TN:
            colsum = torch.full((M,), float("nan"), device="cuda")
            got = matmul(fwp._lib, TN, x, y, colsum=colsum)
            assert bool(((got.double() - raw).abs() <= bound(K, mag)).all())
            assert bool(((colsum.double() - a.sum(1)).abs() <= K * EPS * a.abs().sum(1)).all())
        got = matmul(fwp._lib, layout, x, y, bias=bias, relu=1, residual=residual, gate=gate)
        assert bool(((got.double() - want).abs() <= bound(K, mag + 400)).all())


@pytest.mark.parametrize("rows", [40, 2100])
@pytest.mark.parametrize("odd", [-1, -99, -101, 300, 2 ** 32 + 5, -2 ** 40])
def test_a_target_that_is_no_word(fwp, odd, rows):
    """-100 is ignored; any other number outside the vocabulary shows as NaN in its loss and in the gradients."""
    x, W, b = randn(rows, 64, seed=1), randn(300, 64, seed=2) * 0.1, randn(300, seed=3)
    target = torch.randint(0, 300, (rows,), generator=torch.Generator().manual_seed(4)).cuda()
    target[3] = -100
    check_loss(fwp._lib, x, W, b, target)
    target[7] = odd
    loss, gx, gW, gb = loss_and_gradients(fwp._lib, x, W, b, target, randn(rows, seed=5))
    assert torch.nonzero(loss.isnan()).flatten().tolist() == [7] and float(loss[3]) == 0
    assert torch.nonzero(gx.isnan().any(1)).flatten().tolist() == [7]
    assert bool(gW.isnan().all()) and bool(gb.isnan().all())


@pytest.mark.parametrize("M,N,K", [(70, 66, 200), (300, 260, 1100), (40, 64, 2048), (2100, 2100, 40)])
@pytest.mark.parametrize("layout", [NT, NN, TN])
def test_products_of_infinities_and_the_largest_numbers(fwp, layout, M, N, K):
    """Operands that bf16 cannot hold (infinities, NaN, numbers above its largest) meet the others as in fp32."""
    A = randn(*((K, M) if layout == TN else (M, K)), seed=1)
    B = randn(*((N, K) if layout == NT else (K, N)), seed=2)
    a, b = (A.t() if layout == TN else A), (B.t() if layout == NT else B)
    inf, big = float("inf"), 3.4e38            # rounds to infinity as a bf16 number
    a[0, 3], a[1, K - 1], a[2, 0], a[3, 5], a[4, 7] = inf, -inf, float("nan"), big, -big
    b[4, 0], b[K - 2, 1] = inf, float("nan")
    b[3, 2], b[5], b[7] = 0.0, 0.01, -0.01     # infinity * 0; results that fp32 holds
    want = a.double() @ b.double()
    mag = a.double().abs() @ b.double().abs()
    for cut in (True, False):
        got = matmul(fwp._lib, layout, A, B, cut).double()
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        assert bool((got == want)[want.isinf()].all())
        ok = want.isfinite()
        assert bool(((got - want).abs() <= (bound(K, mag) + K * EPS * mag))[ok].all())      # K roundings in a row


def test_loss_gradients_of_an_infinite_upstream_gradient(fwp):
    x, W, b = randn(40, 64, seed=1), randn(300, 64, seed=2) * 0.1, randn(300, seed=3)
    target = torch.randint(0, 300, (40,), generator=torch.Generator().manual_seed(4)).cuda()
    gloss = randn(40, seed=5)
    gloss[7] = float("inf")
    _, *got = loss_and_gradients(fwp._lib, x, W, b, target, gloss)
    xd, Wd, bd = (t.double().requires_grad_() for t in (x, W, b))
    want = torch.nn.functional.cross_entropy(xd @ Wd.t() + bd, target, reduction="none")
    for name, g, w in zip("xWb", got, torch.autograd.grad(want, (xd, Wd, bd), gloss.double())):
        odd = ~w.isfinite()      # at the target PyTorch forms infinity - p infinity, NaN, and (p - 1) infinity is also right
        assert torch.equal(~g.isfinite(), odd) and bool((g == w)[w.isinf()].all()), name
        assert float((g.double() - w)[~odd].abs().max() if bool((~odd).any()) else 0.0) <= 2e-5 * 10, name


# 64 x 64 (all at once, cut or not; step by step), 128 x 64 and 128 x 128 tiles, k in ranges; B's rows kept in LDS (4 and 8 steps of k, whole and not)
HALF_SHAPES = [(70, 130, 128), (3, 5, 131), (65, 66, 256), (200, 70, 257), (64, 64, 2111), (8190, 509, 300), (2100, 3001, 260), (131, 776, 3001), (6433, 1030, 131), (6433, 1030, 200),
               (3201, 2048, 256)]


@pytest.mark.parametrize("M,N,K", HALF_SHAPES)
@pytest.mark.parametrize("layout", [NT, NN, TN])
@pytest.mark.parametrize("case", ["even", "growing", "sparse"])
def test_products_of_two_fp16_parts(fwp, M, N, K, layout, case):
    """Rows of the same size throughout, rows that grow along k far beyond fp16's range (up and down again), rows of zeros
    with a few elements; with every epilogue, operands apart and unaligned."""
    a, b = randn(M, K, seed=1), randn(N, K, seed=2)
    if case == "growing":
        step = torch.arange(K, device="cuda") / K
        a = a * torch.exp2(60 * step - 40) * torch.exp2(20 * randn(M, 1, seed=6))
        b = b * torch.exp2(40 * (0.5 - (step - 0.5).abs()))
    elif case == "sparse":
        a, b = a * (randn(M, K, seed=6) > 2), b * (randn(N, K, seed=7) > 2) * 1e-20
        a[M // 2], b[N // 2] = 0, 0
    bias, residual, gate = randn(N, seed=3), randn(M, N, seed=4), randn(M, N, seed=5)
    x, y = a.double(), b.double()
    raw, mag = x @ y.t(), x.abs() @ y.abs().t()
    err = bound(K, mag)
    A, B = a.t().contiguous() if layout == TN else a, b if layout == NT else b.t().contiguous()
    for by, first in ((0, 0), (3, 1)):
        p, q = spread(A, by, first), spread(B, by, first)
        assert bool(((matmul(fwp._lib, layout, p, q).double() - raw).abs() <= err).all())
        got = matmul(fwp._lib, layout, p, q, bias=bias, relu=1, residual=residual, gate=gate)
        want = torch.where(gate > 0, torch.relu(raw + bias.double()) + residual.double(), 0.0)
        assert bool(((got.double() - want).abs() <= err + 2 * EPS * (raw.abs() + bias.abs() + residual.abs())).all())


@pytest.mark.parametrize("M,N,K", [(8190, 509, 300), (6433, 1030, 200), (3201, 2048, 128), (1000, 70, 200), (1000, 130, 700)])
@pytest.mark.parametrize("layout", [NT, NN, TN])
def test_infinities_in_larger_products(fwp, M, N, K, layout):
    a, b = randn(M, K, seed=1), randn(N, K, seed=2)
    a[7, 3], a[M - 1, K - 1], a[900, 0], b[N - 1, 5] = float("inf"), float("nan"), 2e37, float("inf")
    a[39], a[40] = 0, a[40] * 2.0 ** (-24 * (torch.arange(K, device="cuda") % 5 == 0))      # an infinity alone beside small elements
    a[39, 3] = float("inf")
    want, mag = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    A, B = a.t().contiguous() if layout == TN else a, b if layout == NT else b.t().contiguous()
    got = matmul(fwp._lib, layout, A, B).double()
    assert torch.equal(got.isnan(), want.isnan()) and bool((got == want)[want.isinf()].all())
    ok = want.isfinite()
    assert bool(((got - want).abs() <= bound(K, mag) + K * EPS * mag)[ok].all())


def wide_operands(case, M, N, K):
    """Operands whose rows hold elements of very different sizes, the large ones against zeros of the other operand."""
    a, b = randn(M, K, seed=1), randn(N, K, seed=2)
    if case in ("outlier", "weight"):          # one large element a row (the other operand has zeros there), of growing size
        x, y = (a, b) if case == "outlier" else (b, a)
        x[:, K // 3] = torch.exp2(torch.linspace(8, 110, len(x), device="cuda"))
        y[:, K // 3] = 0
    elif case == "late":                       # the same at the end of k, 2^20 above the rest: scales change at the last moment
        a[:, K - 1], b[:, K - 1] = 2.0 ** 20, 0
        b[:, K - 2], a[:, K - 2] = 2.0 ** 20, 0
    elif case == "groups":                     # a third of the features 2^18 times as large, with zeros for weights; and the reverse
        a[:, ::3] *= 2.0 ** 18
        b[:, ::3] = 0
        b[:, 1::3] *= 2.0 ** 18
        a[:, 1::3] = 0
    elif case == "picked":                     # every result is one element of a
        a = a * torch.exp2(-40 * torch.rand(M, K, generator=torch.Generator().manual_seed(3)).cuda())
        b = torch.nn.functional.one_hot(torch.arange(N, device="cuda") * 7 % K, K).float()
    elif case == "even":                       # sizes over 2^40 in both, half of them zeros: many small elements
        r = lambda i, *s: torch.rand(*s, generator=torch.Generator().manual_seed(i)).cuda()
        a = a * torch.exp2(-40 * r(3, M, K)) * (r(4, M, K) < 0.5)
        b = b * torch.exp2(-40 * r(5, N, K)) * (r(6, N, K) < 0.5)
    elif case in ("spread", "weights"):        # every k of one operand has a size of its own, over 2^56 (beyond the second time of small elements)
        x = a if case == "spread" else b
        x *= torch.exp2(-56 * torch.rand(K, generator=torch.Generator().manual_seed(3)).cuda())
    elif case == "few":                        # small elements now and then: too few to give up on fp16
        a[:, ::41] *= 2.0 ** -24
        b[:, 7::97] *= 2.0 ** -30
    return a, b


@pytest.mark.parametrize("M,N,K", HALF_SHAPES)
@pytest.mark.parametrize("layout", [NT, NN, TN])
@pytest.mark.parametrize("case", ["outlier", "weight", "late", "groups", "picked", "even", "spread", "weights", "few"])
def test_rows_of_elements_of_very_different_sizes(fwp, M, N, K, layout, case):
    """An element counts to its own size, whatever else is in its row."""
    a, b = wide_operands(case, M, N, K)
    x, y = a.double(), b.double()
    want, mag = x @ y.t(), x.abs() @ y.abs().t()
    A, B = a.t().contiguous() if layout == TN else a, b if layout == NT else b.t().contiguous()
    for cut in (True, False):
        got = matmul(fwp._lib, layout, A, B, cut).double()
        assert bool(((got - want).abs() <= bound(K, mag)).all())


@pytest.mark.parametrize("M,N,K,layout", [(256, 1024, 32768, TN), (32768, 256, 1024, NT), (32768, 1024, 256, NT), (256, 128, 2000, TN)])
def test_sizes_that_are_spread_cost_no_multiple(fwp, M, N, K, layout):
    """Where every k has a size of its own (tokens' gradients; features) three bf16 numbers' six products take over from three, or
    three more are made: twice the time, and something for the change.  (Element by element: 6 to 9 times.)"""
    def microseconds(A, B):
        matmul(fwp._lib, layout, A, B)
        times = []
        for _ in range(9):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(10):
                matmul(fwp._lib, layout, A, B)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return sorted(times)[4]

    a, b = randn(M, K, seed=1), randn(N, K, seed=2)
    sizes = torch.exp(5 * randn(K, seed=3))
    A, S = (a.t().contiguous(), (a * sizes).t().contiguous()) if layout == TN else (a, a * sizes)
    B = b if layout == NT else b.t().contiguous()
    assert microseconds(S, B) <= 3.5 * microseconds(A, B)


@pytest.mark.parametrize("rows,vocab", [(70, 300), (6500, 6600)])
def test_logits_of_an_outlying_feature(fwp, rows, vocab):
    """A feature 2^20 above the others whose weights are zero: the losses are those without it."""
    L, dim = fwp._lib, 132
    x, W, b = randn(rows, dim, seed=1), randn(vocab, dim, seed=2) * 0.3, randn(vocab, seed=3)
    x[:, 5], W[:, 5] = 2.0 ** 20, 0
    target = torch.randint(0, vocab, (rows,), generator=torch.Generator().manual_seed(4)).cuda()
    loss = loss_and_gradients(L, x, W, b, target, randn(rows, seed=5))[0]
    want = torch.nn.functional.cross_entropy(x.double() @ W.double().t() + b.double(), target, reduction="none")
    err = bound(dim, x.double().abs() @ W.double().abs().t() + b.double().abs()).max() + 2.0 ** -20
    assert float((loss.double() - want).abs().max()) <= float(err)


@pytest.mark.parametrize("rows,cols", [(1, 4), (5, 36), (3000, 128), (2500, 256), (9, 260), (70, 1024)])
def test_layer_norm(fwp, rows, cols):
    L = fwp._lib
    x, g, b, gy = (randn(*s, seed=i) for i, s in enumerate(((rows, cols), (cols,), (cols,), (rows, cols))))
    x = 3 * x + 1
    xd, gd, bd = (t.double().requires_grad_() for t in (x, g, b))
    want = torch.nn.functional.layer_norm(xd, (cols,), gd, bd, 1e-5)
    wants = torch.autograd.grad(want, (xd, gd, bd), gy.double())
    y, stats = torch.full_like(x, float("nan")), torch.empty(rows, 2, device="cuda")
    assert L.lib().fwp_layer_norm_fwd(x.data_ptr(), g.data_ptr(), b.data_ptr(), y.data_ptr(), stats.data_ptr(), rows, cols,
                                      1e-5, L.stream_of(x)) == 0
    # cols roundings in a sum, a few more around it, of values whose scale is that of the row
    tol = (cols / 8 + 16) * EPS
    rms = xd.detach().abs().max() / xd.detach().std(-1, keepdim=True, correction=0).clamp_min(1e-2)
    assert bool(((y.double() - want).abs() <= tol * rms * (gd.abs() + 1) * 4 + 1e-6).all())
    gx, gg, gb = torch.full_like(x, float("nan")), torch.empty_like(g), torch.empty_like(b)
    work = torch.empty(L.lib().fwp_layer_norm_workspace(rows, cols), device="cuda")
    assert L.lib().fwp_layer_norm_bwd(gy.data_ptr(), x.data_ptr(), stats.data_ptr(), g.data_ptr(),
                                      gx.data_ptr(), gg.data_ptr(), gb.data_ptr(), work.data_ptr(), rows, cols,
                                      L.stream_of(x)) == 0
    for name, got, w in zip(("x", "gamma", "beta"), (gx, gg, gb), wants):
        scale = float(w.abs().max()) + float(gy.abs().max())
        assert float((got.double() - w).abs().max()) <= (rows / 8 + cols / 8 + 64) * EPS * scale * float(rms.max()), name


# tiles of 256 columns and of 128 in one range of k, with a rest of k and of columns; an infinity in an operand
@pytest.mark.parametrize("rows,vocab,dim", [(4100, 4133, 1408), (5501, 5500, 1406)])
@pytest.mark.parametrize("odd", [False, True])
def test_gradients_from_an_operand_split_once(fwp, rows, vocab, dim, odd):
    """With a workspace the loss's gradients read their second operand split beforehand, without one they split it: the same numbers."""
    L = fwp._lib
    x, W, b = randn(rows, dim, seed=1) * 0.1, randn(vocab, dim, seed=2) * 0.3, randn(vocab, seed=3)
    target = torch.randint(0, vocab, (rows,), generator=torch.Generator().manual_seed(4)).cuda()
    gloss = randn(rows, seed=5)
    logits, loss, stats = torch.empty(rows, vocab, device="cuda"), torch.empty(rows, device="cuda"), torch.empty(rows, 2, device="cuda")
    work = torch.empty(L.lib().fwp_nll_workspace(rows, vocab), device="cuda")
    s = L.stream_of(x)
    assert L.lib().fwp_nll_stats_fwd(x.data_ptr(), W.data_ptr(), b.data_ptr(), target.data_ptr(), logits.data_ptr(), loss.data_ptr(),
                                     stats.data_ptr(), work.data_ptr(), rows, vocab, dim, s) == 0
    if odd:
        x[rows - 1, 3] = W[70, dim - 1] = float("inf")
    n = max(L.lib().fwp_matmul_workspace(rows, dim, vocab), L.lib().fwp_matmul_workspace(vocab, dim, rows))
    assert n > 3 * dim * rows // 2
    work = torch.full((n + 64,), 7.0, device="cuda")
    results = []
    for w in (work.data_ptr(), None):
        out = [torch.full_like(t, 5.0) for t in (x, W, b)]
        assert L.lib().fwp_nll_stats_bwd(x.data_ptr(), W.data_ptr(), logits.data_ptr(), stats.data_ptr(), target.data_ptr(),
                                         gloss.data_ptr(), *(t.data_ptr() for t in out), w, rows, vocab, dim, s) == 0
        results.append(out)
    assert bool((work[n:] == 7).all())
    for a, c in zip(*results):
        assert bool(((a == c) | (a.isnan() & c.isnan())).all()) and bool(a.isfinite().all()) != (odd and a is not results[0][2])


def test_gradients_off_a_16_byte_boundary_leave_the_rest_of_the_workspace(fwp):
    """Such results get another plan than the one the workspace's size comes from: nothing behind that size is written, and the numbers are those
    of a call without a workspace."""
    L = fwp._lib
    rows, vocab, dim = 10142, 35166, 258
    x, W, b = randn(rows, dim, seed=1) * 0.1, randn(vocab, dim, seed=2) * 0.3, randn(vocab, seed=3)
    target = torch.randint(0, vocab, (rows,), generator=torch.Generator().manual_seed(4)).cuda()
    gloss = randn(rows, seed=5)
    logits, loss, stats = torch.empty(rows, vocab, device="cuda"), torch.empty(rows, device="cuda"), torch.empty(rows, 2, device="cuda")
    work = torch.empty(L.lib().fwp_nll_workspace(rows, vocab), device="cuda")
    s = L.stream_of(x)
    assert L.lib().fwp_nll_stats_fwd(x.data_ptr(), W.data_ptr(), b.data_ptr(), target.data_ptr(), logits.data_ptr(), loss.data_ptr(),
                                     stats.data_ptr(), work.data_ptr(), rows, vocab, dim, s) == 0
    n = max(L.lib().fwp_matmul_workspace(rows, dim, vocab), L.lib().fwp_matmul_workspace(vocab, dim, rows))
    work = torch.full((n + (8 << 20),), 7.0, device="cuda")
    results = []
    for w in (work.data_ptr(), None):
        out = [torch.full((t.numel() + 1,), 5.0, device="cuda") for t in (x, W, b)]
        assert L.lib().fwp_nll_stats_bwd(x.data_ptr(), W.data_ptr(), logits.data_ptr(), stats.data_ptr(), target.data_ptr(),
                                         gloss.data_ptr(), *(t.data_ptr() + 4 for t in out), w, rows, vocab, dim, s) == 0
        assert all(float(t[0]) == 5.0 for t in out)
        results.append(out)
    assert bool((work[n:] == 7).all())
    assert all(torch.equal(a, c) for a, c in zip(*results))


@pytest.mark.parametrize("layout,M,N,K", [(NT, 16, 256, 4096), (TN, 776, 256, 3001), (NN, 257, 36, 1000), (TN, 130, 70, 9000), (TN, 4100, 256, 4100)])
def test_a_product_stays_within_its_own_workspace(fwp, layout, M, N, K):
    """Its size leaves out what only the loss's gradients use; the partial sums are those of a call with room for both."""
    L = fwp._lib
    A, B = randn(*((K, M) if layout == TN else (M, K)), seed=1), randn(*((N, K) if layout == NT else (K, N)), seed=2)
    n = L.lib().fwp_product_workspace(M, N, K)
    assert 0 <= n <= L.lib().fwp_matmul_workspace(M, N, K)
    work, C = torch.full((n + 4096,), 7.0, device="cuda"), torch.empty(M, N, device="cuda")
    colsum = torch.empty(M, device="cuda")
    e = L.Epilogue(None, None, None, colsum.data_ptr() if layout == TN else None, 0)
    assert L.lib().fwp_matmul(layout, A.data_ptr(), A.stride(0), B.data_ptr(), B.stride(0), C.data_ptr(), N, M, N, K, ctypes.byref(e),
                              work.data_ptr(), L.stream_of(A)) == 0
    assert bool((work[n:] == 7).all())
    assert torch.equal(C, matmul(L, layout, A, B))
