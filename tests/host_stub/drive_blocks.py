"""Drives the language model's blocks (csrc/fwp_torch_blocks.cpp) in the host build (see build.sh) on host tensors, against
the same computation by PyTorch's operators in float64: the stand-in library computes the products, LayerNorm and the
loss, so what is compared is what the blocks make of them.  Run as a script (python drive_blocks.py BUILD_DIR CHECK),
normally by tests/test_binding_host.py.  Prints 'CHECK ok' at the end."""
import importlib
import os
import sys

import torch
import torch.nn.functional as F

from drive import load, rnd

TOL = 2e-5          # fp32 results of double sums of a few hundred terms of size one


def close(got, want, what):
    got, want = got.detach().double(), want.detach().double()
    assert got.shape == want.shape, (what, got.shape, want.shape)
    err, size = float((got - want).abs().max()), float(want.abs().max())
    assert err <= TOL * (1 + size), (what, err, size)


def compare(ours, ref, args, what):
    """A block and its reference on the same arguments: result, and gradients of those that want one."""
    a = [t.clone().requires_grad_(t.requires_grad) if torch.is_tensor(t) and t.is_floating_point() else t for t in args]
    b = [t.detach().double().requires_grad_(t.requires_grad) if torch.is_tensor(t) and t.is_floating_point() else t
         for t in args]
    y, want = ours(*a), ref(*b)
    close(y, want, what)
    g = torch.randn_like(y)
    wants = [t for t in b if torch.is_tensor(t) and t.requires_grad]
    got = torch.autograd.grad(y, [t for t in a if torch.is_tensor(t) and t.requires_grad], g)
    for i, (x, z) in enumerate(zip(got, torch.autograd.grad(want, wants, g.double()))):
        close(x, z, (what, i))
    with torch.no_grad():
        close(ours(*args), want, what)


def linear_of(x, W, b=None, relu=False):
    y = F.linear(x, W, b)
    return torch.relu(y) if relu else y


def feed_forward_of(x, W1, b1, W2, b2, residual=None):
    y = F.linear(torch.relu(F.linear(x, W1, b1)), W2, b2)
    return y if residual is None else y + residual


def nll_of(x, W, b, target):
    return F.cross_entropy(F.linear(x, W, b), target, reduction="none")


def unaligned(t):
    """The same values 4 bytes off a 16-byte boundary."""
    buf = torch.empty(t.numel() + 4)
    first = (-buf.data_ptr() // 4) % 4 + 1
    out = buf[first:first + t.numel()].view(t.shape)
    out.copy_(t.detach())
    assert out.data_ptr() % 16 == 4 and out.is_contiguous()
    return out.requires_grad_(t.requires_grad)


def results(m):
    """Every block, inputs contiguous, permuted and off a 16-byte boundary, gradients wanted in part."""
    W, b = rnd(24, 64, grad=True), rnd(24, grad=True)
    for x in (rnd(7, 3, 64, grad=True), rnd(3, 70, 64).transpose(0, 1).requires_grad_(), unaligned(rnd(90, 64, grad=True)), rnd(64)):
        for bias, relu in ((b, False), (b, True), (None, False), (None, True)):
            compare(m.linear, linear_of, (x, W, bias, relu), "linear")
    compare(m.linear, linear_of, (rnd(5, 64, grad=True), W.detach(), b), "linear, weight frozen")
    compare(m.linear, linear_of, (rnd(5, 64), unaligned(W), None), "linear, weight off a boundary")
    W1, b1, W2, b2 = rnd(40, 24, grad=True), rnd(40, grad=True), rnd(24, 40, grad=True), rnd(24, grad=True)
    for x in (rnd(9, 2, 24, grad=True), unaligned(rnd(5, 24, grad=True)), rnd(24, 6).t().requires_grad_()):
        compare(m.feed_forward, feed_forward_of, (x, W1, b1, W2, b2), "feed-forward")
        compare(m.feed_forward, feed_forward_of, (x, W1, b1, W2, b2, rnd(*x.shape, grad=True)), "with a residual")
        compare(lambda x, *p: m.feed_forward(x, *p, x), lambda x, *p: feed_forward_of(x, *p, x), (x, W1, b1, W2, b2), "its input added")
    compare(m.feed_forward, feed_forward_of, (rnd(4, 24), W1.detach(), b1, W2, b2.detach()), "some frozen")
    g, z = rnd(24, grad=True), rnd(24, grad=True)
    for x in (rnd(6, 24, grad=True), rnd(2, 3, 24, grad=True).transpose(0, 1), rnd(3, 24)):
        compare(lambda x, g, z: m.layer_norm(x, g, z, 1e-5), lambda x, g, z: F.layer_norm(x, (24,), g, z, 1e-5), (x, g, z), "LayerNorm")
    target = torch.tensor([3, 0, -100, 23, 7])
    compare(m.nll, nll_of, (rnd(5, 64, grad=True), W, b, target), "loss")
    compare(m.nll, nll_of, (rnd(5, 64), W, b.detach(), target), "loss, hidden state frozen")
    ids = torch.randint(0, 24, (4, 3))
    freq = rnd(32).abs()
    phase = torch.arange(3.0, -1, -1).clamp_max(2)[:, None] * freq
    want = W[ids] * 8.0 + torch.cat((phase.sin(), phase.cos()), -1)[:, None]
    close(m.embed(W, ids, freq, 8.0, 2.0), want, "embedding")


def refused(f, *args):
    for grad in (True, False):
        with torch.set_grad_enabled(grad):
            try:
                f(*args)
            except (RuntimeError, AssertionError):
                continue
        raise AssertionError(("accepted", f, [tuple(t.shape) for t in args if torch.is_tensor(t)]))


def misfits(m):
    """Operands whose sizes do not fit one another raise before a kernel gets their addresses."""
    x, W, b, W2, b2 = rnd(6, 64, grad=True), rnd(128, 64, grad=True), rnd(128), rnd(64, 128), rnd(64)
    for bad in ((rnd(6, 60), W, b), (rnd(6, 128), W, b), (x, W, rnd(127)), (x, W, rnd(129)), (x, rnd(128), None), (rnd(()), W, None)):
        refused(m.linear, *bad)
    refused(m.feed_forward, rnd(6, 32), W, b, W2, b2)
    refused(m.feed_forward, x, W, b, rnd(64, 96), b2)           # 8192 of 6144 floats
    refused(m.feed_forward, x, W, b, rnd(64, 130), b2)
    refused(m.feed_forward, x, W, rnd(120), W2, b2)
    refused(m.feed_forward, x, W, b, W2, rnd(60))
    refused(m.feed_forward, x, W, b, W2, b2, rnd(1, 64))
    refused(m.feed_forward, x, W, b, rnd(1, 128), rnd(1))
    target = torch.zeros(6, dtype=torch.int64)
    for bad in ((x, rnd(100, 32), rnd(100)), (x, rnd(100, 64), rnd(90)), (x, rnd(100, 65), rnd(100)), (x, rnd(100, 64), rnd(101))):
        refused(m.nll, *bad, target)
    refused(m.nll, x, rnd(100, 64), rnd(100), target[:5])
    refused(m.nll, rnd(2, 3, 64), rnd(100, 64), rnd(100), target)
    for bad in ((rnd(6, 24), rnd(24), rnd(20)), (rnd(6, 24), rnd(20), rnd(20)), (rnd(6, 24), rnd(28), rnd(24)), (rnd(6, 24), rnd(2, 12), rnd(24))):
        refused(m.layer_norm, *bad, 1e-5)
    y, Wqkvb, Wo, state = rnd(5, 2, 48, grad=True), rnd(3 * 49, 48), rnd(48, 48), torch.zeros(2, 3, 16, 16)
    m.delta_block(y, Wqkvb, Wo, state, 3, 16, 0.25, True)
    for bad in ((y, Wqkvb, rnd(40, 48), state), (y, Wqkvb, rnd(50, 48), state), (y, Wqkvb, rnd(48, 32), state), (y, rnd(146, 48), Wo, state),
                (y, rnd(3 * 49, 40), Wo, state), (y, Wqkvb, Wo, torch.zeros(1, 3, 16, 16)), (rnd(10, 48), Wqkvb, Wo, state)):
        refused(m.delta_block, *bad, 3, 16, 0.25, True)
    refused(m.embed, rnd(24, 64), torch.zeros(4, 3, dtype=torch.int64), rnd(30), 8.0, 0.0)
    refused(m.embed, rnd(24, 64), torch.zeros(4, dtype=torch.int64), rnd(32), 8.0, 0.0)
    refused(m.embed, rnd(64), torch.zeros(4, 3, dtype=torch.int64), rnd(32), 8.0, 0.0)


class Recorded:
    """The blocks, with the names of those that were called."""

    def __init__(self, m):
        self.m, self.calls = m, []

    def __getattr__(self, name):
        f = getattr(self.m, name)
        if name.startswith("takes_"):
            return f

        def call(*args):
            self.calls.append(name)
            return f(*args)
        return call

    def of(self, f, *args):
        """The blocks that f(*args) goes through, and its result (an exception among them)."""
        self.calls.clear()
        try:
            res = f(*args)
        except Exception as e:
            res = e
        return list(self.calls), res


def package(m):
    """The package with its layers on the host build's blocks: host tensors count as the GPU's, and the operator that
    stands in for fast_weight_delta in a layer's general path returns its values."""
    sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))
    pkg = importlib.import_module("recurrent-fwp_amd")
    layers, rec = pkg.layers, Recorded(m)
    layers._fwp_torch = rec
    layers.fast_weight_delta = lambda q, k, v, beta, W, *more: v
    return pkg, rec


def misfitting_modules(m):
    """Modules whose parameters do not fit one another do what they do on stock PyTorch."""
    pkg, rec = package(m)
    nn, x = torch.nn, rnd(5, 2, 24)
    ff = pkg.PositionwiseFF(24, 40, 0.0)
    assert rec.of(ff, x)[0] == ["feed_forward", "layer_norm"]
    ff.CoreNet[3] = nn.Linear(40, 1)                       # added to the input by broadcasting
    calls, y = rec.of(ff._core, x, x)
    assert calls == [] and torch.equal(y, x + ff.CoreNet(x))
    ff.CoreNet[3] = nn.Linear(36, 24)
    calls, e = rec.of(ff, x)
    assert calls == [] and type(e) is RuntimeError, e
    ff = pkg.PositionwiseFF(24, 40, 0.0)
    for bad in (rnd(5, 2, 20), rnd(5, 2, 48)):
        calls, e = rec.of(ff, bad)
        assert calls == [] and type(e) is RuntimeError, e
    crit, target = pkg.lm._TiedSoftmaxLoss(100, 24), torch.zeros(6, dtype=torch.int64)
    assert rec.of(crit, rnd(6, 24), target)[0] == ["nll"]
    for hidden, t in ((rnd(6, 20), target), (rnd(6, 30), target), (rnd(6, 24), target[:5])):
        calls, e = rec.of(crit, hidden, t)
        assert calls in ([], ["linear"]) and type(e) in (RuntimeError, ValueError), e
    calls, y = rec.of(crit, rnd(24), target[0])            # one token without a batch
    assert calls == ["linear"] and y.shape == ()
    crit.out_layers[0].weight = nn.Parameter(rnd(120, 24))  # a vocabulary that grew without its bias
    calls, e = rec.of(crit, rnd(6, 24), target)
    assert calls == [] and type(e) is RuntimeError, e
    lin = pkg.layers.Linear(24, 0)
    calls, y = rec.of(lin, x)
    assert calls == [] and y.shape == (5, 2, 0)


def language_model(pkg, rec, **more):
    """A small model that decodes on the host build: its input, and the first state of every layer."""
    pkg.lm.DeltaNetLM._embed = lambda self, data: self.word_emb(data).detach() if not torch.is_grad_enabled() else None
    lm = pkg.DeltaNetLM(**{**dict(n_token=50, n_layer=3, n_head=4, d_model=64, d_head=16, d_inner=64), **more})
    toks = torch.randint(0, 50, (1, 3))
    with torch.no_grad():
        calls, (hid, mems) = rec.of(lambda: lm.hidden(toks, None, carry_over_fast_weight=True))
    assert calls == ["decode_layers"] and len(mems) == 3
    return lm, toks, mems


def decode(rec, lm, toks, mems):
    with torch.no_grad():
        calls, res = rec.of(lambda: lm.hidden(toks, mems, carry_over_fast_weight=True))
    if isinstance(res, Exception):
        raise res
    return calls, res


def states_left_out(m):
    """None in the place of a layer's state is no state, as for the layers one by one."""
    pkg, rec = package(m)
    lm, toks, mems = language_model(pkg, rec)
    for given in ([None] * 3, [mems[0], None, mems[2]]):
        calls, (hid, new) = decode(rec, lm, toks, given)
        assert "decode_layers" not in calls and calls.count("delta_block") == 3 and len(new) == 3


def unusual_parameters(m):
    """Weights that are plain attributes (replicas, flattened parameters) or off a 16-byte boundary, modules left out."""
    pkg, rec = package(m)
    nn = torch.nn
    lm, toks, mems = language_model(pkg, rec)
    want = decode(rec, lm, toks, mems)[1][0]
    for lin in (lm.layers[1].dec_attn.qkvb_net, lm.layers[1].pos_ff.CoreNet[0], lm.layers[2].pos_ff.layer_norm):
        w = lin.weight.detach().clone()
        del lin.weight
        lin.weight = w
        calls, (hid, _) = decode(rec, lm, toks, mems)
        assert calls == ["decode_layers"] and torch.equal(hid, want)
    lin = lm.layers[1].pos_ff.CoreNet[3]
    lin.weight = nn.Parameter(unaligned(lin.weight))
    calls, _ = decode(rec, lm, toks, mems)
    assert calls.count("delta_block") == 3 and calls.count("feed_forward") == 3, calls
    lin.weight = nn.Parameter(lin.weight.detach().clone())
    assert decode(rec, lm, toks, mems)[0] == ["decode_layers"]
    lm.layers[1].pos_ff.CoreNet[0].bias = None
    calls, _ = decode(rec, lm, toks, mems)
    assert "decode_layers" not in calls and calls.count("delta_block") == 3

    class Other(nn.Module):             # a layer of another kind, first
        def forward(self, x, mems=None, carry_over_fast_weight=False):
            return x, mems
    lm, toks, mems = language_model(pkg, rec)
    lm.layers[0] = Other()
    calls, _ = decode(rec, lm, toks, mems)
    assert "decode_layers" not in calls and calls.count("delta_block") == 2


def wrapped_modules(m):
    """A sub-module whose forward was replaced on the instance (adapters, instrumentation) is called."""
    pkg, rec = package(m)

    def wrap(mod):
        inner, seen = mod.forward, []

        def forward(*args, **kwargs):
            seen.append(1)
            return inner(*args, **kwargs)
        mod.forward = forward
        return seen

    x = rnd(5, 2, 24)
    for pick in (lambda f: f.CoreNet, lambda f: f.CoreNet[0], lambda f: f.CoreNet[1], lambda f: f.CoreNet[4], lambda f: f.layer_norm):
        ff = pkg.PositionwiseFF(24, 40, 0.0)
        seen = wrap(pick(ff))
        ff(x)
        assert seen == [1]
    crit = pkg.lm._TiedSoftmaxLoss(30, 24)
    seen = wrap(crit.out_layers[0])
    crit(rnd(6, 24), torch.zeros(6, dtype=torch.int64))
    assert seen == [1]
    for pick in (lambda l: l, lambda l: l.dec_attn, lambda l: l.pos_ff, lambda l: l.pos_ff.CoreNet[3], lambda l: l.pos_ff.layer_norm,
                 lambda l: l.dec_attn.drop, lambda l: l.dec_attn.layer_norm):
        lm, toks, mems = language_model(pkg, rec)
        seen = wrap(pick(lm.layers[1]))
        decode(rec, lm, toks, mems)
        assert seen == [1], pick


def replaced_dropouts(m):
    """The model's dropout replaced or hooked: it runs on the embedding and on the last hidden state, in both modes."""
    pkg, rec = package(m)
    nn = torch.nn

    class Half(nn.Module):
        def forward(self, x):
            return 0.5 * x
    for training in (True, False):
        lm, toks, mems = language_model(pkg, rec)
        lm.train(training)
        lm.drop = nn.Identity()
        decode(rec, lm, toks, mems)
        seen = []
        lm.drop = nn.Dropout(0.0)
        lm.drop.register_forward_hook(lambda *a: seen.append(1))
        decode(rec, lm, toks, mems)
        assert seen == [1, 1]
        lm.drop = Half()
        calls, (hid, _) = decode(rec, lm, toks, mems)
        with torch.no_grad():
            want = lm._through_layers(0.5 * lm._embed(toks), mems, True)[0]
        assert "decode_layers" not in calls and torch.equal(hid, want)


def own_scales(m):
    """A layer's read-out scale is its attribute, when all layers decode in one call too."""
    pkg, rec = package(m)
    lm, toks, mems = language_model(pkg, rec)
    hidden = decode(rec, lm, toks, mems)[1][0]
    for layer in lm.layers:
        layer.dec_attn.scale = 0.5
    calls, (hid, _) = decode(rec, lm, toks, mems)
    assert calls == ["decode_layers"] and not torch.equal(hid, hidden)
    for other in (0.125, torch.tensor(0.5)):
        lm.layers[1].dec_attn.scale = other
        assert decode(rec, lm, toks, mems)[0].count("delta_block") == 3


def states_of_their_own(m):
    """A layer's carried state has its own memory: keeping one keeps no other."""
    pkg, rec = package(m)
    lm, toks, mems = language_model(pkg, rec)
    for W, _ in mems:
        assert W.untyped_storage().nbytes() == W.numel() * 4 and W.is_contiguous()


def replaced_states(m):
    """What a layer starts from comes from its _state, replaced on the instance, in a subclass or on the class."""
    pkg, rec = package(m)
    cls = pkg.layers.DeltaNetLayer
    H, D, x = 2, 16, rnd(5, 3, 32)
    layer = cls(H, 32, D)
    with torch.no_grad():
        zero = layer(x, carry_over_fast_weight=True)[1][0]

    def other(self, mems, carry_over_fast_weight, bsz, h, dtype):
        return torch.full((bsz, H, D, D), 0.5, dtype=dtype)

    class Sub(cls):
        _state = other

    sub = Sub(H, 32, D)
    sub.load_state_dict(layer.state_dict())
    here = cls(H, 32, D)
    here.load_state_dict(layer.state_dict())
    here._state = lambda *a: other(None, *a)
    own = cls._state
    try:
        for mod in (sub, here, layer):
            if mod is layer:
                cls._state = other
            with torch.no_grad():
                calls, (_, (W, _)) = rec.of(lambda: mod(x, carry_over_fast_weight=True))
            assert calls.count("delta_block") == 1 and float((W - zero).abs().max()) > 0.1, type(mod)
    finally:
        cls._state = own


def beyond_the_kernels(m):
    """Matrices wider than the kernels' offsets reach (2^21) and inputs of more rows than a launch takes go to PyTorch."""
    pkg, rec = package(m)
    crit, wide = pkg.lm._TiedSoftmaxLoss(5, 2), 2 ** 21 + 1
    crit.out_layers[0] = pkg.layers.Linear(2, wide)
    with torch.no_grad():
        calls, loss = rec.of(crit, rnd(3, 2), torch.zeros(3, dtype=torch.int64))
        assert calls == [] and loss.shape == (3,)
        calls, y = rec.of(pkg.layers.Linear(wide, 2), rnd(1, wide))
        assert calls == [] and y.shape == (1, 2)
        ff = pkg.PositionwiseFF(2, wide, 0.0)
        calls, y = rec.of(ff, rnd(1, 2))
        assert calls == [] and y.shape == (1, 2)
    x = torch.empty(1, 1).expand(2 ** 24 + 1, 4)           # no memory behind it
    assert not m.takes_linear(x, rnd(4, 4), rnd(4)) and m.takes_linear(x[:2 ** 24], rnd(4, 4), rnd(4))
    assert not m.takes_all(x, [rnd(4)]) and m.takes_all(x[:2 ** 24], [rnd(4)])


def traced_and_watched(m):
    """Tracers, the script compiler and modes that watch the operators see PyTorch's; a default device changes nothing."""
    from torch.fx.experimental.proxy_tensor import make_fx
    pkg, rec = package(m)
    x, target = rnd(6, 24), torch.randint(0, 30, (6,))

    class Watch(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, f, types, args=(), kwargs=None):
            return f(*args, **(kwargs or {}))

    class WatchFunctions(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, f, types, args=(), kwargs=None):
            return f(*args, **(kwargs or {}))

    for mod, args in ((pkg.PositionwiseFF(24, 40, 0.0), (x,)), (pkg.PositionwiseFF(24, 40, 0.0, True), (x,)),
                      (pkg.layers.Linear(24, 9), (x,)), (pkg.lm._TiedSoftmaxLoss(30, 24), (x, target))):
        with torch.no_grad():
            calls, want = rec.of(mod, *args)
            assert calls
            with torch.device("cpu"):
                assert rec.of(mod, *args)[0] == calls
            others = (torch.fx.symbolic_trace(mod), torch.jit.script(mod), torch.jit.trace(mod, args),
                      make_fx(lambda *a: mod(*a))(*args), torch.compile(mod, backend="eager", fullgraph=True))
            for other in others:
                calls, y = rec.of(other, *args)
                assert calls in ([], ["linear"]) and torch.allclose(y, want, atol=1e-5), (type(mod), other, y)
            for mode in (Watch, WatchFunctions):
                with mode():
                    calls, y = rec.of(mod, *args)
                assert calls == [] and torch.allclose(y, want, atol=1e-5)


def main():
    m, check = load(sys.argv[1]), sys.argv[2]
    torch.manual_seed(0)
    globals()[check](m)
    print(check + " ok")


if __name__ == "__main__":
    main()
