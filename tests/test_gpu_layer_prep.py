"""The Delta-Net layer's pre-step and its adjoint where a workgroup's rows (eight heads of consecutive steps) are cut: few and many heads,
single steps, odd numbers of sequences, rows at every alignment, against float64."""
import importlib

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def layers():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return importlib.import_module("recurrent-fwp_amd.layers")


def oracle(x, H, D, scale):
    q, k, v, b = x.view(*x.shape[:2], H, 3 * D + 1).split([D, D, D, 1], -1)
    f = torch.nn.functional.elu(q) + 1, torch.nn.functional.elu(k) + 1
    q, k = (z / z.sum(-1, keepdim=True) for z in f)
    return [z.permute(1, 2, 0, 3) for z in (q * scale, k, v, b.sigmoid())]


@pytest.mark.parametrize("T,B,H,D", [(1, 1, 1, 16), (1, 7, 20, 32), (33, 5, 3, 16), (7, 3, 9, 16), (64, 20, 1, 64), (5, 2, 8, 64),
                                     (3, 1, 12, 32), (130, 3, 8, 32), (31, 9, 2, 32)])
def test_rows(layers, T, B, H, D):
    torch.manual_seed(T + B)
    x = torch.randn(T, B, H * (3 * D + 1), device="cuda", requires_grad=True)
    ref = x.detach().double().cpu().requires_grad_()
    got, want = layers.DeltaNetPrep.apply(x, H, D, 0.25), oracle(ref, H, D, 0.25)
    grads = [torch.randn_like(g) for g in got]
    got[0].sum()        # results may be read before the adjoint runs
    dx, = torch.autograd.grad(got, x, grads)
    dref, = torch.autograd.grad(want, ref, [g.double().cpu() for g in grads])
    # An entry is rounded at most about eight times, the exponential (2^-22) and a sum of D included: 2^-20 of it.  In the adjoint of q
    # and k two terms of that error cancel; their size is at most that of v's and beta's gradients beside them.
    for a, b in list(zip(got, want)) + [(dx, dref)]:
        assert a.shape == b.shape
        assert float((a.double().cpu() - b).norm()) <= 2 ** -20 * float(b.norm())


@pytest.mark.parametrize("rows,cols", [(1, 4), (3, 60), (17, 64), (16, 68), (15, 128), (33, 132), (8193, 256), (8, 260), (8191, 64),
                                       (9001, 4), (20001, 60), (1025, 68), (2003, 96), (1030, 128), (8197, 132), (10243, 188), (16389, 252)])
def test_norm_rows(layers, rows, cols):
    """LayerNorm where a workgroup's rows (4, or 16 of up to 256 columns), a row's last lanes and the workgroups' second turn are cut; with few rows, and with
    those from which on 16 lanes take a row, forward and in the adjoint."""
    L = importlib.import_module("recurrent-fwp_amd._lib")
    torch.manual_seed(rows + cols)
    x, gy = torch.randn(2, rows, cols, device="cuda")
    g, b = torch.randn(2, cols, device="cuda")
    ref = [z.double().cpu().requires_grad_() for z in (x, g, b)]
    want = torch.nn.functional.layer_norm(ref[0], (cols,), ref[1], ref[2], 1e-5)
    refs = torch.autograd.grad(want, ref, gy.double().cpu())
    y, gx, stats, gg, gb = torch.empty_like(x), torch.empty_like(x), torch.empty(rows, 2, device="cuda"), torch.empty_like(g), torch.empty_like(b)
    s = torch.cuda.current_stream().cuda_stream
    L.check(L.lib().fwp_layer_norm_fwd(x.data_ptr(), g.data_ptr(), b.data_ptr(), y.data_ptr(), stats.data_ptr(), rows, cols, 1e-5, s), "fwd")
    work = torch.empty(L.lib().fwp_layer_norm_workspace(rows, cols), device="cuda")
    L.check(L.lib().fwp_layer_norm_bwd(gy.data_ptr(), x.data_ptr(), stats.data_ptr(), g.data_ptr(), gx.data_ptr(), gg.data_ptr(), gb.data_ptr(),
                                       work.data_ptr(), rows, cols, s), "bwd")
    # about eight roundings an entry (sums of up to 64 lane shares among them): 2^-20 of the result; the column sums add up to rows / 8192
    # rounded terms a lane and 64 shares one after the other: well below 2^-18
    for got, ref, bound in ((y, want, 2 ** -20), (gx, refs[0], 2 ** -20), (gg, refs[1], 2 ** -18), (gb, refs[2], 2 ** -18)):
        assert float((got.double().cpu() - ref).norm()) <= bound * float(ref.norm())


@pytest.mark.parametrize("cols", [60, 64, 68, 128, 132, 192, 252, 256])
def test_norm_of_a_row_does_not_depend_on_the_number_of_rows(layers, cols):
    """More rows take 16 lanes each instead of 64: every number is the same to the last bit, results and gradients of x."""
    L = importlib.import_module("recurrent-fwp_amd._lib")
    torch.manual_seed(cols)
    rows, few = 16400, 100
    x, gy = torch.randn(2, rows, cols, device="cuda")
    g, b = torch.randn(2, cols, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    got = []
    for n in (rows, few):
        y, gx, stats, gg, gb = torch.empty_like(x[:n]), torch.empty_like(x[:n]), torch.empty(n, 2, device="cuda"), torch.empty_like(g), torch.empty_like(b)
        L.check(L.lib().fwp_layer_norm_fwd(x.data_ptr(), g.data_ptr(), b.data_ptr(), y.data_ptr(), stats.data_ptr(), n, cols, 1e-5, s), "fwd")
        work = torch.empty(L.lib().fwp_layer_norm_workspace(n, cols), device="cuda")
        L.check(L.lib().fwp_layer_norm_bwd(gy.data_ptr(), x.data_ptr(), stats.data_ptr(), g.data_ptr(), gx.data_ptr(), gg.data_ptr(), gb.data_ptr(),
                                           work.data_ptr(), n, cols, s), "bwd")
        got.append((y[:few], stats[:few], gx[:few]))
    assert all(torch.equal(a, c) for a, c in zip(*got))


@pytest.mark.parametrize("T,B,D", [(1, 3, 16), (5, 2, 64), (40, 9, 32)])
def test_a_fresh_state_starts_at_zero(layers, T, B, D):
    """Fewer lanes than the state has groups, and more; whatever the state's memory held."""
    L = importlib.import_module("recurrent-fwp_amd._lib")
    H = 3
    x = torch.randn(T, B, H * (3 * D + 1), device="cuda")
    state = torch.full((B * H * D * D + 8,), float("nan"), device="cuda")
    a, b = ([torch.empty(B, H, T, n, device="cuda") for n in (D, D, D, 1)] for _ in range(2))
    s = torch.cuda.current_stream().cuda_stream
    L.check(L.lib().fwp_deltanet_prep_start(x.data_ptr(), *(t.data_ptr() for t in a), state.data_ptr(), T, B, H, D, 0.5, s), "start")
    L.check(L.lib().fwp_deltanet_prep_fwd(x.data_ptr(), *(t.data_ptr() for t in b), T, B, H, D, 0.5, s), "fwd")
    assert not bool(state[:-8].any()) and bool(state[-8:].isnan().all())
    assert all(torch.equal(p, q) for p, q in zip(a, b))
