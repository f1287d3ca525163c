"""The layers on the C++ blocks against themselves in float64 on stock PyTorch: dropout in and out, LayerNorm
before and after, hooks and second derivatives (which take stock PyTorch), products in every order."""
import pytest
import torch

from oracle.torch_loop import delta_loop

pytestmark = pytest.mark.gpu


def loop_op(q, k, v, beta, W):
    out, W_end = delta_loop(q, k, v, beta, W.clone())
    W.copy_(W_end.detach())
    return out


def close(name, got, want, scale=1.0):
    """A few dozen fp32 roundings of values of the size of `want`."""
    got, want = got.detach(), want.detach()
    err, size = (got.double() - want).abs().max(), want.abs().max()
    assert float(err) <= 64 * 2.0 ** -24 * float(size) * scale, f"{name}: {float(err):.2e} of {float(size):.2e}"


def both(make, x, seed=0):
    """The module in fp32 and in float64 with the same parameters, and their input."""
    torch.manual_seed(seed)
    ours, ref = make(None).cuda(), make(loop_op).cuda().double()
    with torch.no_grad():
        for p in ours.parameters():
            p.normal_(0.0, 0.2)
    ref.load_state_dict(ours.state_dict())
    return ours, ref, x.clone().requires_grad_(), x.double().requires_grad_()


@pytest.mark.parametrize("drop", [0.0, 1e-9])       # 1e-9: the path with dropout, nothing dropped
@pytest.mark.parametrize("pre", [False, True])
def test_feed_forward_block(fwp, pre, drop):
    x = torch.randn(37, 3, 64, generator=torch.Generator().manual_seed(1)).cuda()
    ours, ref, a, b = both(lambda op: fwp.PositionwiseFF(64, 200, drop, pre), x)
    y, want = ours(a), ref(b)
    close("y", y, want)
    g = torch.randn_like(x)
    grads = torch.autograd.grad(y, [a, *ours.parameters()], g)
    wants = torch.autograd.grad(want, [b, *ref.parameters()], g.double())
    for i, (got, w) in enumerate(zip(grads, wants)):
        close(i, got, w, 4)


@pytest.mark.parametrize("drop", [0.0, 1e-9])
@pytest.mark.parametrize("pre,D", [(False, 16), (True, 32), (False, 64)])
def test_delta_block(fwp, pre, D, drop):
    x = torch.randn(50, 3, 96, generator=torch.Generator().manual_seed(1)).cuda()
    ours, ref, a, b = both(lambda op: fwp.DeltaNetLayer(2, 96, D, dropout=drop, pre_lnorm=pre, fast_weight_op=op), x)
    W0 = torch.randn(3, 2, D, D, generator=torch.Generator().manual_seed(2)).cuda() * 0.1
    y, (W, _) = ours(a, mems=(W0, None), carry_over_fast_weight=True)
    want, (W_want, _) = ref(b, mems=(W0.double(), None), carry_over_fast_weight=True)
    close("y", y, want)
    close("W", W, W_want)
    g = torch.randn_like(x)
    grads = torch.autograd.grad(y, [a, *ours.parameters()], g)
    wants = torch.autograd.grad(want, [b, *ref.parameters()], g.double())
    for i, (got, w) in enumerate(zip(grads, wants)):
        close(i, got, w, 16)
    # frozen weights, an input that wants nothing
    for p in ours.parameters():
        p.requires_grad_(False)
    ours.o_net.weight.requires_grad_(True)
    y, _ = ours(x, mems=(W0, None), carry_over_fast_weight=True)
    got, = torch.autograd.grad(y, [ours.o_net.weight], g)
    assert torch.equal(got, grads[1 + [n for n, _ in ours.named_parameters()].index("o_net.weight")])


def test_second_derivatives_and_hooks_take_stock_operators(fwp):
    x = torch.randn(9, 2, 32, generator=torch.Generator().manual_seed(1)).cuda()
    ours, ref, a, b = both(lambda op: fwp.PositionwiseFF(32, 64, 0.0), x)
    seconds = []
    for m, z in ((ours, a), (ref, b)):
        g, = torch.autograd.grad(m(z).square().sum(), [z], create_graph=True)
        seconds.append(torch.autograd.grad(g.square().sum(), [z, *m.parameters()], allow_unused=True))
    for i, (got, want) in enumerate(zip(*seconds)):
        assert (got is None) == (want is None)
        if got is not None:
            close(i, got, want, 64)
    seen = []
    ours.CoreNet[1].register_forward_hook(lambda m, i, o: seen.append(o.shape))
    ours(a)
    assert seen == [(9, 2, 64)]


@pytest.mark.parametrize("pre", [False, True])
@pytest.mark.parametrize("power", [1, 2])
def test_second_derivatives_of_the_delta_block(fwp, pre, power):
    """Through the gradients of every parameter and of the input, as from the layer's general path (a hook on the dropout
    sends it there): the delta rule's own gradients are constants there, what they are multiplied with is not."""
    x, c = torch.randn(2, 20, 2, 48, generator=torch.Generator().manual_seed(1)).cuda()      # c: a sum over LayerNorm is constant
    seconds = []
    for general in (False, True):
        torch.manual_seed(0)
        m = fwp.DeltaNetLayer(3, 48, 16, pre_lnorm=pre).cuda()
        if general:
            m.drop.register_forward_hook(lambda *a: None)
        z = x.clone().requires_grad_()
        firsts = torch.autograd.grad(((c * m(z)) ** power).sum(), [z, *m.parameters()], create_graph=True)
        # one by one: what each first derivative depends on
        g = torch.Generator().manual_seed(2)
        for (name, _), first in zip([("x", z), *m.named_parameters()], firsts):
            w = torch.randn(first.shape, generator=g).cuda()
            if first.requires_grad:
                got = torch.autograd.grad((first * w).sum(), [z, *m.parameters()], allow_unused=True, retain_graph=True)
            else:
                got = [None] * len(firsts)
            seconds += [(general, name, i, t) for i, t in enumerate(got)]
    half = len(seconds) // 2
    for (_, name, i, got), (_, _, _, want) in zip(seconds[:half], seconds[half:]):
        zero = torch.zeros(1, device="cuda")      # no dependence and a gradient of zeros are the same
        got, want = zero if got is None else got, zero if want is None else want.double()
        if got.numel() == 1 or want.numel() == 1:
            assert float(got.abs().max()) == float(want.abs().max()) == 0, (name, i)
        else:
            close((name, i), got, want, 64)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_decoder_layer_under_autocast(fwp, dtype):
    """PyTorch's products in the lower precision around the fp32 operator."""
    x = torch.randn(20, 2, 64, generator=torch.Generator().manual_seed(1)).cuda().requires_grad_()
    torch.manual_seed(0)
    layer = fwp.DeltaNetDecoderLayer(2, 64, 32, 128).cuda()
    w = torch.randn_like(x)
    want = layer(x)
    wants = torch.autograd.grad((want * w).sum(), [x, *layer.parameters()])
    with torch.autocast("cuda", dtype=dtype):
        y = layer(x)
    grads = torch.autograd.grad((y * w).sum(), [x, *layer.parameters()])
    # four products of bf16's 8 bits in a row.  In the 2-norm: an activation that rounding takes across the ReLU's zero
    # changes single elements of a gradient by a token's whole share (one of 40 tokens here, up to 2 ** -3 of the largest).
    for got, ref in zip((y, *grads), (want, *wants)):
        assert got.dtype is torch.float32 and float((got - ref).norm()) <= 16 * 2.0 ** -8 * float(ref.norm())


@pytest.mark.parametrize("pre", [False, True])
def test_language_model_with_ignored_targets(fwp, pre):
    """Losses and every gradient of a two-layer model, some targets ignored, frozen embedding included."""
    cfg = dict(n_token=309, n_layer=2, n_head=3, d_model=48, d_head=16, d_inner=100, pre_lnorm=pre, tie_weight=False)
    torch.manual_seed(0)
    ours = fwp.DeltaNetLM(init_std=0.3, **cfg).cuda()
    ref = fwp.DeltaNetLM(fast_weight_op=loop_op, init_std=0.3, **cfg).cuda().double()
    ref.load_state_dict(ours.state_dict())
    g = torch.Generator().manual_seed(1)
    data, target = (torch.randint(0, 309, (45, 3), generator=g).cuda() for _ in range(2))
    target[5:9, 1] = -100
    (loss,), (want,) = ours(data, target), ref(data, target)
    close("loss", loss, want)
    assert bool((loss[5:9, 1] == 0).all())
    with torch.no_grad():
        close("loss without a graph", ours(data, target)[0], want)
    w = torch.randn(45, 3, generator=g).cuda()
    (loss * w).sum().backward()
    (want * w.double()).sum().backward()
    for (name, a), (_, b) in zip(ours.named_parameters(), ref.named_parameters()):
        close(name, a.grad, b.grad, 16)


@pytest.mark.parametrize("B,D,dm,inner,pre", [(1, 16, 128, 64, False), (5, 32, 128, 192, True), (17, 32, 256, 2048, False),
                                              (33, 64, 1024, 128, True), (64, 16, 64, 1088, False), (50, 16, 64, 64, True),
                                              (65, 16, 128, 64, False)])       # 65: the layers one by one
def test_decoding_one_token_at_a_time(fwp, B, D, dm, inner, pre):
    """Hidden states, logits and carried states of three tokens, the first without a state, against float64."""
    cfg = dict(n_token=150, n_layer=2, n_head=4, d_model=dm, d_head=D, d_inner=inner, pre_lnorm=pre)
    torch.manual_seed(0)
    ours = fwp.DeltaNetLM(init_std=0.2, **cfg).cuda()
    ref = fwp.DeltaNetLM(fast_weight_op=loop_op, init_std=0.2, **cfg).cuda().double()
    ref.load_state_dict(ours.state_dict())
    toks = torch.randint(0, 150, (3, 1, B), generator=torch.Generator().manual_seed(1)).cuda()
    mems = mems_ref = None
    with torch.no_grad():
        for t in toks:
            hid, mems = ours.hidden(t, mems, carry_over_fast_weight=True)
            want, mems_ref = ref.hidden(t, mems_ref, carry_over_fast_weight=True)
            close("hidden", hid, want)
            close("logits", ours.crit.out_layers[0](hid), ref.crit.out_layers[0](want))
            for (W, _), (W_ref, _) in zip(mems, mems_ref):
                close("state", W, W_ref)
        assert torch.equal(ours.hidden(toks[0])[0], ours.hidden(toks[0], carry_over_fast_weight=True)[0])


def same_nans(name, got, want):
    assert torch.equal(got.isnan(), want.isnan()), name
    ok = ~want.isnan()
    if bool(ok.any()):
        close(name, got[ok], want[ok], 16)


# tiles of whole 16-byte groups and others; a k in one range and in several
@pytest.mark.parametrize("rows,d,inner", [(40, 64, 200), (40, 66, 201), (300, 512, 1024)])
@pytest.mark.parametrize("where", ["W1", "b1", "x"])
def test_nan_passes_the_feed_forward_blocks_relu(fwp, where, rows, d, inner):
    """torch.relu(NaN) is NaN, and its gradient passes where the activation is NaN."""
    x = torch.randn(rows, 1, d, generator=torch.Generator().manual_seed(1)).cuda()
    ours, ref, a, b = both(lambda op: fwp.PositionwiseFF(d, inner, 0.0, True), x)
    nan = float("nan")
    with torch.no_grad():
        for m, z in ((ours, a), (ref, b)):
            {"W1": m.CoreNet[0].weight, "b1": m.CoreNet[0].bias[None], "x": z[0]}[where][0, 3] = nan
    # without LayerNorm in between, which would spread a NaN of x over its row
    ours.layer_norm, ref.layer_norm = torch.nn.Identity(), torch.nn.Identity()
    y, want = ours(a), ref(b)
    same_nans("y", y, want)
    g = torch.randn_like(x)
    grads = torch.autograd.grad(y, [a, *ours.parameters()], g)
    wants = torch.autograd.grad(want, [b, *ref.parameters()], g.double())
    for i, (got, w) in enumerate(zip(grads, wants)):
        same_nans(i, got, w)


@pytest.mark.parametrize("B", [3, 20, 40])
def test_nan_passes_the_decoding_paths_relu(fwp, B):
    cfg = dict(n_token=50, n_layer=1, n_head=4, d_model=64, d_head=16, d_inner=128)
    torch.manual_seed(0)
    ours = fwp.DeltaNetLM(init_std=0.2, **cfg).cuda()
    ours.layers[0].pos_ff.CoreNet[0].bias.data[5] = float("nan")
    with torch.no_grad():
        hid, _ = ours.hidden(torch.zeros(1, B, dtype=torch.int64, device="cuda"))
        assert bool(hid.isnan().all())
        z = torch.randn(B, 1, 64, device="cuda")
        lin = ours.layers[0].pos_ff.CoreNet[0]
        same_nans("few rows", fwp._fwp_torch.linear(z, lin.weight, lin.bias, True), torch.relu(lin(z)).double())


@pytest.mark.parametrize("T,clamp", [(1, -1), (300, -1), (70, 20)])
def test_embedding_without_a_graph(fwp, T, clamp):
    """The fused embedding against the lines it replaces (they run when a graph is recorded)."""
    lm = fwp.DeltaNetLM(n_token=50, n_layer=1, n_head=2, d_model=36, d_head=16, d_inner=32, clamp_len=clamp).cuda()
    lm.layers = torch.nn.ModuleList()
    data = torch.randint(0, 50, (T, 3), generator=torch.Generator().manual_seed(1)).cuda()
    want, _ = lm.hidden(data)
    with torch.no_grad():
        got, _ = lm.hidden(data)
    assert float((got - want.detach()).abs().max()) <= 2.0 ** -22
