"""Drives the language model's blocks (csrc/fwp_torch_blocks.cpp) in the host build (see build.sh) on host tensors, against
the same computation by PyTorch's operators in float64: the stand-in library computes the products, LayerNorm and the
loss, so what is compared is what the blocks make of them.  Run as a script (python drive_blocks.py BUILD_DIR CHECK),
normally by tests/test_binding_host.py.  Prints 'CHECK ok' at the end."""
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


def main():
    m, check = load(sys.argv[1]), sys.argv[2]
    torch.manual_seed(0)
    globals()[check](m)
    print(check + " ok")


if __name__ == "__main__":
    main()
