"""The delta rule over few long sequences, which are cut into segments that run at the same time."""
import numpy as np
import pytest
import torch

import oracle
from helpers import delta_inputs, within

pytestmark = pytest.mark.gpu

# N, H, L, E, M: the shortest that is cut, a last segment of one step, of whole blocks, key widths of each kernel
SHAPES = [(1, 8, 640, 32, 32), (1, 1, 641, 32, 16), (2, 3, 1281, 16, 16), (1, 5, 1408, 16, 32), (2, 2, 700, 16, 64), (1, 2, 1000, 64, 16),
          (1, 2, 777, 64, 64), (1, 3, 900, 96, 16), (2, 1, 830, 96, 32), (1, 2, 650, 32, 64), (8, 8, 1000, 32, 32)]


@pytest.mark.parametrize("N,H,L,E,M", SHAPES)
@pytest.mark.parametrize("steps_first", [False, True])
def test_segments_against_the_oracle(fwp, N, H, L, E, M, steps_first):
    assert fwp._lib.lib().fwp_delta_segment_floats(N, H, L, E, M, 64) > 0
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
