"""The delta rule over few long sequences, which are cut into segments that run at the same time."""
import numpy as np
import pytest
import torch

import oracle
from helpers import delta_inputs, within

pytestmark = pytest.mark.gpu

# N, H, L, E, M: the shortest that is cut, a last segment of one step, of whole blocks, key widths of each kernel; values in slices of columns
SHAPES = [(1, 8, 640, 32, 32), (1, 1, 641, 32, 16), (2, 3, 1281, 16, 16), (1, 5, 1408, 16, 32), (2, 2, 700, 16, 64), (1, 2, 1000, 64, 16),
          (1, 2, 777, 64, 64), (1, 3, 900, 96, 16), (2, 1, 830, 96, 32), (1, 2, 650, 32, 64), (8, 8, 1000, 32, 32),
          (1, 2, 900, 64, 32), (1, 1, 1200, 32, 16), (1, 2, 1200, 96, 97)]


@pytest.mark.parametrize("N,H,L,E,M", SHAPES)
@pytest.mark.parametrize("steps_first", [False, True])
def test_segments_against_the_oracle(fwp, N, H, L, E, M, steps_first):
    assert fwp._lib.lib().fwp_delta_segment_floats(N, H, L, E, M if M % 16 == 0 else 16, 64) > 0
    *x, W0, go = delta_inputs(3, N, H, L, E, M, np.float32, w0=True)
    dev = lambda a: (torch.from_numpy(a).permute(2, 0, 1, 3).contiguous().cuda().permute(1, 2, 0, 3) if steps_first
                     else torch.from_numpy(a).cuda())
    ts = [dev(a).requires_grad_(True) for a in x]
    W = torch.from_numpy(W0).cuda()
    out = fwp.fast_weight_delta(*ts, W)
    grads = torch.autograd.grad(out, ts, dev(go))
    double = [a.astype("float64") for a in (*x, W0)]
    want = [*oracle.delta_fwd(*double)[:2], *oracle.delta_bwd(*double, go.astype("float64"))]
    for name, got, w in zip(("out", "W", "q", "k", "v", "beta"), (out, W, *grads), want):
        assert within(got.detach().cpu().numpy(), w, 1e-4, 1e-5), name
    # nothing saved: the same numbers; in pieces: the state goes on
    W1 = torch.from_numpy(W0).cuda()
    with torch.no_grad():
        assert torch.equal(fwp.fast_weight_delta(*ts, W1), out) and torch.equal(W1, W)
        W2 = torch.from_numpy(W0).cuda()
        pieces = [fwp.fast_weight_delta(*(t[:, :, a:b] for t in ts), W2) for a, b in ((0, 17), (17, L))]
    assert within(torch.cat(pieces, 2).cpu().numpy(), want[0], 1e-4, 1e-5) and within(W2.cpu().numpy(), want[1], 1e-4, 1e-5)


def run(fwp, arrays, cut, chunk=64, kind=None):
    """Forward and backward through the C ABI, cut or whole; `kind`: of the forward kernels (the backward ones are chosen)."""
    L_ = fwp._lib
    lib = L_.lib()
    q, k, v, beta, W0, go = (torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda() for a in arrays)
    N, H, L, E = q.shape
    M = v.shape[-1]
    view = lambda t: L_.View(t.data_ptr(), t.stride(0), t.stride(1), t.stride(2))
    W, out, vdiff, gv = W0.clone(), torch.empty_like(v), torch.empty_like(v), torch.empty_like(v)
    ckpt = torch.ones(L_.delta_ckpt_floats(N, H, L, E, M, chunk), device="cuda")
    gq, gk, gb = torch.empty_like(q), torch.empty_like(k), torch.empty_like(beta)
    n = lib.fwp_delta_segment_floats(N, H, L, E, M, chunk)
    assert n > 0
    work = torch.full((n,), float("nan"), device="cuda") if cut else None
    w, dims, stream = (L_.ptr(work) if cut else None), (N, H, L, E, M, chunk), L_.stream_of(q)
    try:
        L_.config(L_.CFG_DELTA_KERNELS, L_.DELTA_AUTO if kind is None else kind)
        L_.check(lib.fwp_delta_fwd_segments(view(q), view(k), view(v), view(beta), L_.ptr(W),
                                            L_.OutView(out.data_ptr(), *out.stride()[:3]), L_.ptr(vdiff), L_.ptr(ckpt), w, *dims, stream), "fwd")
        if cut:
            work.fill_(float("nan"))
    finally:
        L_.config(L_.CFG_DELTA_KERNELS, L_.DELTA_AUTO)
    L_.check(lib.fwp_delta_bwd_segments(view(q), view(k), view(beta), L_.ptr(vdiff), view(go), L_.ptr(ckpt), L_.ptr(gq), L_.ptr(gk),
                                        L_.ptr(gv), L_.ptr(gb), w, *dims, stream), "bwd")
    return dict(zip(("out", "W", "q", "k", "v", "beta"), (t.cpu().numpy() for t in (out, W, gq, gk, gv, gb))))


def oracle_of(arrays):
    x = [np.asarray(a, np.float32).astype(np.float64) for a in arrays]
    return dict(zip(("out", "W", "q", "k", "v", "beta"), [*oracle.delta_fwd(*x[:5])[:2], *oracle.delta_bwd(*x)]))


@pytest.mark.parametrize("N,H,L,E,M", [(1, 8, 2048, 16, 16), (1, 4, 2048, 32, 32), (1, 2, 1500, 64, 32), (1, 2, 1400, 96, 16)])
@pytest.mark.parametrize("keys", ["unit", "half", "weak"])
def test_segments_that_forget(fwp, N, H, L, E, M, keys):
    """Keys of unit norm forget the state before: a large one carried in, and the gradient that comes in at the end.  Every stretch of 64 steps
    to its own size, as precise as whole sequences are: twice their error (they round once a block, segments in their own
    blocks and in the maps of those before) and a rounding's worth.  half: only half of the directions are ever written;
    weak: nothing is forgotten."""
    g = np.random.default_rng(5)
    k, q = (g.standard_normal((N, H, L, E)) for _ in range(2))
    if keys == "half":
        k[..., E // 2:] = 0
    k /= np.linalg.norm(k, axis=-1, keepdims=True)
    beta = 1 / (1 + np.exp(-g.standard_normal((N, H, L, 1)) + (6 if keys == "weak" else 0)))
    go = g.standard_normal((N, H, L, M))
    go[:, :, :-70] = 0
    arrays = (q / np.sqrt(E), k, g.standard_normal((N, H, L, M)), beta, 1e3 * g.standard_normal((N, H, E, M)), go)
    arrays = [a.astype(np.float32) for a in arrays]
    want = oracle_of(arrays)
    cut, whole = run(fwp, arrays, True), run(fwp, arrays, False)
    for name, w in want.items():
        steps = range(0, L, 64) if name != "W" else (0,)
        top = np.linalg.norm(w)
        for t in steps:
            part = (lambda a: a) if name == "W" else (lambda a: a[:, :, t:t + 64])
            size = np.linalg.norm(part(w))
            if size <= 1e-12 * top:
                continue
            err = lambda got: np.linalg.norm(part(got[name]) - part(w)) / size
            assert err(cut) <= 2 * err(whole) + 3e-7, (name, t, err(cut), err(whole))


def test_segments_in_a_graph(fwp):
    """Captured and replayed several times, eager calls between."""
    *x, W0, go = delta_inputs(4, 1, 8, 1000, 32, 32, np.float32, w0=True)
    ts = [torch.from_numpy(a).cuda() for a in x]
    start, W = torch.from_numpy(W0).cuda(), torch.from_numpy(W0).cuda()
    with torch.no_grad():
        want = fwp.fast_weight_delta(*ts, start.clone())
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            fwp.fast_weight_delta(*ts, W)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            W.copy_(start)
            out = fwp.fast_weight_delta(*ts, W)
        for _ in range(4):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            assert torch.equal(fwp.fast_weight_delta(*ts, start.clone()), want)


def test_what_is_cut(fwp):
    floats = lambda *a: fwp._lib.lib().fwp_delta_segment_floats(*a, 64)
    assert floats(1, 8, 639 - 15, 32, 32) == 0 and floats(8, 8, 2048, 32, 32) > 0 and floats(9, 8, 2048, 32, 32) == 0
    assert floats(1, 8, 1264, 16, 16) == 0 and floats(16, 8, 2048, 16, 16) > 0 and floats(17, 8, 2048, 16, 16) == 0
    assert floats(1, 8, 4096, 128, 16) == 0 and floats(1, 8, 4096, 24, 24) == 0 and floats(0, 8, 4096, 16, 16) == -1


def test_backward_is_cut_on_its_own(fwp):
    """Forward and backward are cut from other lengths on; what forward's scratch holds is enough for backward."""
    lib = fwp._lib.lib()
    fwd, bwd = lib.fwp_delta_segment_floats, lib.fwp_delta_bwd_segment_floats
    for E in (16, 32, 64, 96):
        for M in (16, 32, 64):
            for seqs in (1, 8, 32, 64, 100):
                for L in range(600, 1400, 16):
                    assert 0 <= bwd(1, seqs, L, E, M, 64) <= fwd(1, seqs, L, E, M, 64)
    assert fwd(1, 8, 768, 32, 32, 64) > 0 and bwd(1, 8, 768, 32, 32, 64) == 0 and bwd(1, 8, 832, 32, 32, 64) > 0
    assert bwd(1, 64, 640, 96, 16, 64) > 0


@pytest.mark.parametrize("N,H,L,E,M", [(1, 2, 800, 64, 32), (1, 8, 1000, 32, 32), (1, 2, 1300, 16, 16), (1, 2, 1300, 96, 16)])
@pytest.mark.parametrize("chunk,kind", [(64, "DELTA_SCAN"), (128, "DELTA_AUTO"), (256, "DELTA_AUTO")])
def test_segments_of_other_chunks_and_forward_kernels(fwp, N, H, L, E, M, chunk, kind):
    """Backward in segments behind a forward whose kernels leave no inverses; checkpoints further apart."""
    arrays = delta_inputs(6, N, H, L, E, M, np.float32, w0=True)
    got, want = run(fwp, arrays, True, chunk, getattr(fwp._lib, kind)), oracle_of(arrays)
    for name, w in want.items():
        assert within(got[name], w, 1e-4, 1e-5), name
