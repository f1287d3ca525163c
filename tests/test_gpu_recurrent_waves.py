"""The recurrent operators' kernels for 32 x 32 states, whose sequences are shared by several waves that hand tiles (of 8 or 16 steps) and
single steps to each other, at the lengths and numbers of sequences where that can go wrong, against the float64 oracle."""
import importlib

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from helpers import rec_inputs, rnn_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fwp():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return importlib.import_module("recurrent-fwp_amd")


def dev(x, grad=False):
    return torch.from_numpy(np.asarray(x, np.float32)).cuda().requires_grad_(grad)


def check(name, got, want, steps, sums=1):
    """2-norm of the error over that of the result.  A step rounds an entry of the state, or of its gradient, about four times (2^-24 of it
    each); over the steps that adds up at random, sqrt(4 steps), and products with R and the softmaxes' derivatives may enlarge it a few
    times: 32 sqrt(steps + 8) 2^-24."""
    got, want = got.detach().cpu().numpy().astype(np.float64), np.asarray(want, np.float64)
    assert np.isfinite(got).all(), name
    err = np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-30)
    assert err <= 32 * (steps + 8) ** 0.5 * 2.0 ** -24 * sums, (name, err)


# lengths around the tiles of 8 and 16 steps and the state's checkpoints (64 steps), two and three of those
LENGTHS = (2, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 130, 193)


@pytest.mark.parametrize("N,H,L", [(1, 3, L) for L in LENGTHS] + [(171, 3, 18), (257, 3, 18), (257, 4, 17), (386, 4, 9), (257, 3, 160), (257, 3, 161)])
def test_rec_tiles_and_workgroups(fwp, N, H, L):
    """513 to 768, more than 768, 1024 and 1536 sequences: each division into workgroups, with spare waves in the last one; up to 160 steps and more."""
    x = rec_inputs(L + N, N, H, L, 32, w0=True)
    x, go = x[:-1], x[-1]
    x32 = [np.asarray(a, np.float32) for a in x]
    ts = [dev(a, True) for a in x[:8]]
    W, h = dev(x[8]), dev(x[9])
    out = fwp.rec_update_fwm_tanh(*ts, W, h)
    out.backward(dev(go))
    x64 = [a.astype(np.float64) for a in x32]
    for name, a, b in zip(("out", "W", "h"), (out, W, h), oracle.rec_fwd(*x64)):
        check(name, a, b, L)
    grads = oracle.rec_bwd(*x64, np.asarray(go, np.float32).astype(np.float64))
    for name, t, g in zip("qx kx vx bx R_q R_k R_v r_b".split(), ts, grads):
        check("grad " + name, t.grad, g, L)


@pytest.mark.parametrize("N,H,L", [(1, 3, L) for L in LENGTHS] + [(64, 4, 18), (85, 3, 33), (257, 1, 20), (171, 3, 17)])
def test_rnn_tiles_and_workgroups(fwp, N, H, L):
    """256, 255, 257 and 513 sequences: one and two sequences to a workgroup, a spare place in the last one, fewer waves to a sequence."""
    z, k, v, W0, beta, h0, go = (np.asarray(a, np.float32) for a in rnn_inputs(L + N, N, H, L, 32, w0=True))
    ts = [dev(a, True) for a in (z, k, v, beta)]
    W, h = dev(W0), dev(h0)
    out = fwp.fast_rnn_v2(ts[0], ts[1], ts[2], W, ts[3], h)
    out.backward(dev(go))
    x64 = [a.astype(np.float64) for a in (z, k, v, W0, beta, h0)]
    for name, a, b in zip(("out", "W", "h"), (out, W, h), oracle.rnn_fwd(*x64)):
        check(name, a, b, L)
    for name, t, g in zip("z k v beta".split(), ts, oracle.rnn_bwd(*x64, go.astype(np.float64))):
        check("grad " + name, t.grad, g, L)


def test_rec_without_gradients(fwp):
    x = rec_inputs(5, 3, 2, 21, 32, w0=True)
    with torch.no_grad():
        W, h = dev(x[8]), dev(x[9])
        out = fwp.rec_update_fwm_tanh(*[dev(a) for a in x[:8]], W, h)
    for name, a, b in zip(("out", "W", "h"), (out, W, h), oracle.rec_fwd(*[np.asarray(a, np.float32).astype(np.float64) for a in x[:-1]])):
        check(name, a, b, 21)


def test_rec_where_a_step_looks_for_its_largest_entry(fwp):
    """Columns of |R| of more than 20, up to 90 here: with the input's largest entry alone taken off, exponentials and their sums would overflow.  W
    stays 0 in the first steps' reach of such R, so few steps: each multiplies what an entry is off by the logits' size."""
    x = list(rec_inputs(6, 2, 2, 3, 32, w0=True))
    x[4], x[5] = 4 * np.sqrt(32) * x[4], 4 * np.sqrt(32) * x[5]      # R_q, R_k ~ N(0, 16)
    x64 = [np.asarray(a, np.float32).astype(np.float64) for a in x]
    ts = [dev(a, True) for a in x[:8]]
    W, h = dev(x[8]), dev(x[9])
    out = fwp.rec_update_fwm_tanh(*ts, W, h)
    out.backward(dev(x[10]))
    for name, a, b in zip(("out", "W", "h"), (out, W, h), oracle.rec_fwd(*x64[:-1])):
        check(name, a, b, 3, sums=100)
    for name, t, g in zip("qx kx vx bx R_q R_k R_v r_b".split(), ts, oracle.rec_bwd(*x64)):
        check("grad " + name, t.grad, g, 3, sums=100)


def test_rec_matrices_at_any_address(fwp):
    """The state and the slow weights are read and written 16 bytes at a time from addresses of any float; the floats around the state stay."""
    x = rec_inputs(8, 3, 2, 21, 32, w0=True)

    def off(a):
        a = np.asarray(a, np.float32)
        t = torch.full((a.size + 9,), 7.0, device="cuda")
        t[5:-4] = torch.from_numpy(a.ravel()).cuda()
        return t, t[5:-4].view(a.shape)

    ts = [dev(a, True) for a in x[:4]] + [off(a)[1].requires_grad_() for a in x[4:8]]
    (around, W), (_, h) = off(x[8]), off(x[9])
    out = fwp.rec_update_fwm_tanh(*ts, W, h)
    out.backward(dev(x[10]))
    x64 = [np.asarray(a, np.float32).astype(np.float64) for a in x]
    for name, a, b in zip(("out", "W", "h"), (out, W, h), oracle.rec_fwd(*x64[:-1])):
        check(name, a, b, 21)
    assert bool((around[:5] == 7).all()) and bool((around[-4:] == 7).all())
    for name, t, g in zip("qx kx vx bx R_q R_k R_v r_b".split(), ts, oracle.rec_bwd(*x64)):
        check("grad " + name, t.grad, g, 21)


def test_rec_masked_and_undefined_entries(fwp):
    """-infinity in a row of the logits is a probability of 0; a row of nothing else, NaN or +infinity make that step and what follows NaN."""
    x = rec_inputs(7, 2, 1, 12, 32, w0=True)
    x = [np.asarray(a, np.float32) for a in x]
    x[0][0, 0, 3, ::3] = -np.inf
    x[1][0, 0, 5, 1:] = -np.inf
    x64 = [a.astype(np.float64) for a in x]
    with torch.no_grad():
        out = fwp.rec_update_fwm_tanh(*[dev(a) for a in x[:8]], dev(x[8]), dev(x[9]))
    check("out", out, oracle.rec_fwd(*x64[:-1])[0], 12)
    for bad in (np.nan, np.inf):
        y = [a.copy() for a in x]
        y[1][1, 0, 4, 20] = bad
        with torch.no_grad():
            got = fwp.rec_update_fwm_tanh(*[dev(a) for a in y[:8]], dev(y[8]), dev(y[9])).cpu().numpy()
        assert np.isnan(got[1, 0, 4:]).all() and np.isfinite(got[1, 0, :4]).all() and np.isfinite(got[0]).all()
