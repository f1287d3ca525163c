"""The caller of ``fast_weight_delta`` in language modelling: the Delta-Net layer and the
feed-forward block that follows it, with the module and parameter names of the reference
(language_modeling/src/utils/cuda_fast_weight_layer.py:57-188, utils/model_utils.py:15-67)
so a reference state_dict loads unchanged.  On the GPU, in fp32, a layer is HIP kernels throughout: the
fast-weight operator, the elementwise lines in front of it, and the matrix products with their biases,
ReLU and residual additions (``_fwp_torch``'s blocks).  Everything else - other data types, autocast, the CPU,
sub-modules that were replaced or carry hooks - runs on stock PyTorch around the operator.  A caller may
pass another operator (tests do, to compare against a step-by-step loop); the layer then also takes
the stock-PyTorch form.
"""
import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.utils._device import DeviceContext

from . import _lib
from .fast_weight import _fwp_torch, fast_weight_delta


def _untouched(m, cls):
    """Is this sub-module exactly a ``cls`` (not a replacement) with its class's ``forward``, that nothing is hooked to?"""
    return type(m) is cls and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks
                                   or "forward" in m.__dict__)


def _watched():
    """Does a mode see the operators that are called?  (A default device is such a mode, but changes none of them.)"""
    if torch._C._len_torch_dispatch_stack():
        return True
    return any(type(torch._C._get_function_stack_at(i)) is not DeviceContext for i in range(torch._C._len_torch_function_stack()))


def _blocks(takes, *args):
    """The C++ blocks (csrc/fwp_torch_blocks.cpp) if they apply, else ``None``.  Their function ``takes`` says so of the
    tensors: ordinary ones, fp32, on the GPU, of sizes that fit one another; here: a call outside autocast, tracing, modes and
    functional transforms."""
    if _fwp_torch is None or torch.compiler.is_compiling() or torch.jit.is_tracing() or not getattr(_fwp_torch, takes)(*args):
        return None
    if (torch.is_autocast_enabled() or _watched() or torch.nn.modules.module._has_any_global_hook()
            or torch.autograd.forward_ad._current_level >= 0 or torch._C._functorch.peek_interpreter_stack() is not None):
        return None
    return _fwp_torch


def _drops(m):
    """Does this dropout module change anything now?"""
    return m.training and m.p > 0


class Linear(nn.Linear):
    """``nn.Linear`` on the package's matrix products where they apply."""

    def forward(self, x):
        if torch.jit.is_scripting():
            return F.linear(x, self.weight, self.bias)
        else:
            return self._forward(x)

    def _forward(self, x):
        blocks = _blocks("takes_linear", x, self.weight, self.bias)
        if blocks is not None:
            return blocks.linear(x, self.weight, self.bias)
        return F.linear(x, self.weight, self.bias)


def _own(m, name):
    """A parameter of a module, or the plain tensor in its place (a replica's, a flattened parameter's), or ``None``."""
    p = m._parameters.get(name)
    return p if p is not None else m.__dict__.get(name)


def decode_parameters(layer):
    """The parameters of a :class:`DeltaNetDecoderLayer` as ``decode_layers`` takes them, or ``None`` when the layer
    is not what that function computes: a replaced or hooked sub-module, an active dropout, another operator."""
    if not (_untouched(layer, DeltaNetDecoderLayer)):
        return None
    att, ff = layer._modules.get("dec_attn"), layer._modules.get("pos_ff")
    if not (_untouched(att, DeltaNetLayer) and _untouched(ff, PositionwiseFF)) or att.fast_weight_op is not fast_weight_delta:
        return None
    a, f = att._modules, ff._modules
    net = f.get("CoreNet")
    if not (_untouched(net, nn.Sequential) and len(net._modules) == 5):
        return None
    lin1, relu, drop1, lin2, drop2 = net._modules.values()
    norms, projections = (a.get("layer_norm"), f.get("layer_norm")), (a.get("qkvb_net"), a.get("o_net"))
    for m in (*projections, lin1, lin2):
        if not _untouched(m, nn.Linear):
            return None
    for m in (a.get("drop"), drop1, drop2):
        if not _untouched(m, nn.Dropout) or _drops(m):
            return None
    for m in norms:
        if not _untouched(m, nn.LayerNorm) or m.eps != norms[0].eps:
            return None
    if not _untouched(relu, nn.ReLU) or att.pre_lnorm != ff.pre_lnorm:
        return None
    if any(_own(m, "bias") is not None for m in projections):
        return None
    params = [_own(m, "weight") for m in projections]
    for m in (norms[0], lin1, lin2, norms[1]):
        params += [_own(m, "weight"), _own(m, "bias")]
    return None if any(p is None for p in params) else params


def _layer_norm(m, x):
    """``m(x)`` for a LayerNorm over the last axis."""
    if _untouched(m, nn.LayerNorm) and len(m.normalized_shape) == 1:
        blocks = _blocks("takes_layer_norm", x, m.weight, m.bias, m.normalized_shape[0])
        if blocks is not None:
            return blocks.layer_norm(x, m.weight, m.bias, m.eps)
    return m(x)


class PositionalEmbedding(nn.Module):
    """Sinusoidal embedding of a position sequence: ``[sin | cos]`` halves, shape
    ``[len, 1, demb]`` (or ``[len, bsz, demb]``).  utils/model_utils.py:15-31."""

    def __init__(self, demb):
        super().__init__()
        self.demb = demb
        self.register_buffer("inv_freq", 10000.0 ** (-torch.arange(0.0, demb, 2.0) / demb))

    def forward(self, pos_seq, bsz=None):
        phase = pos_seq[:, None] * self.inv_freq[None, :]
        emb = torch.cat((phase.sin(), phase.cos()), dim=-1).unsqueeze(1)
        return emb if bsz is None else emb.expand(-1, bsz, -1)


class PositionwiseFF(nn.Module):
    """Linear-ReLU-Linear with residual and LayerNorm (after, or before when
    ``pre_lnorm``).  utils/model_utils.py:34-67.  The reference's ReLU works in place; on a
    ``[len, bsz, d_inner]`` input that is a view of the projection's 2-D result, and autograd then
    rebuilds the base tensor in backward (three copies and a clone of the widest activation per
    layer, 4 % of the language model's step): not in place here."""

    def __init__(self, d_model, d_inner, dropout, pre_lnorm=False):
        super().__init__()
        self.d_model, self.d_inner, self.dropout, self.pre_lnorm = d_model, d_inner, dropout, pre_lnorm
        self.CoreNet = nn.Sequential(
            nn.Linear(d_model, d_inner), nn.ReLU(), nn.Dropout(dropout),
            nn.Linear(d_inner, d_model), nn.Dropout(dropout))
        self.layer_norm = nn.LayerNorm(d_model)

    def _core(self, x, residual):
        """``residual + CoreNet(x)``"""
        net = self.CoreNet
        if (_untouched(net, nn.Sequential) and len(net) == 5 and _untouched(net[0], nn.Linear) and _untouched(net[1], nn.ReLU)
                and _untouched(net[2], nn.Dropout) and _untouched(net[3], nn.Linear) and _untouched(net[4], nn.Dropout)):
            W1, b1, W2, b2 = net[0].weight, net[0].bias, net[3].weight, net[3].bias
            blocks = _blocks("takes_feed_forward", x, W1, b1, W2, b2)
            if blocks is not None and not (_drops(net[2]) or _drops(net[4])):
                return blocks.feed_forward(x, W1, b1, W2, b2, residual)
            if blocks is not None:
                hid = net[2](blocks.linear(x, W1, b1, True))
                return residual + net[4](blocks.linear(hid, W2, b2))
        return residual + net(x)

    def forward(self, inp):
        if torch.jit.is_scripting():
            out = inp + self.CoreNet(self.layer_norm(inp) if self.pre_lnorm else inp)
            return out if self.pre_lnorm else self.layer_norm(out)
        else:
            return self._forward(inp)

    def _forward(self, inp):
        if self.pre_lnorm:
            return self._core(_layer_norm(self.layer_norm, inp), inp)
        return _layer_norm(self.layer_norm, self._core(inp, inp))


def sum_normalised_elu(x):
    """``phi(x) = (elu(x) + 1) / sum_D(elu(x) + 1)``: positive features that sum to one
    (cuda_fast_weight_layer.py:118-123)."""
    x = F.elu(x) + 1.0
    return x / x.sum(-1, keepdim=True)


class DeltaNetPrep(torch.autograd.Function):
    """``q, k, v, beta = DeltaNetPrep.apply(qkvb, n_head, d_head[, q_scale])``: the lines between the layer's
    projection and the operator (cuda_fast_weight_layer.py:108-125) as one HIP kernel each way.
    ``qkvb`` is the contiguous ``[len, bsz, n_head * (3 d_head + 1)]`` projection; the results are
    contiguous ``[bsz, n_head, len, .]``: q, k through :func:`sum_normalised_elu`, v copied, beta
    through a sigmoid.  ``q_scale`` multiplies q: the operator's output is linear in q, so the
    ``1/sqrt(d_head)`` the layer applies to that output (:155-157) can ride here for free."""

    @staticmethod
    def supported(qkvb, d_head):
        return (qkvb.is_cuda and qkvb.dtype == torch.float32 and qkvb.is_contiguous()
                and d_head in (16, 32, 64))

    @staticmethod
    def forward(ctx, qkvb, n_head, d_head, q_scale=1.0):
        _lib.require_device(qkvb)
        T, B, _ = qkvb.shape
        H, D = n_head, d_head
        f32 = dict(device=qkvb.device, dtype=torch.float32)
        q, k, v = (torch.empty((B, H, T, D), **f32) for _ in range(3))
        beta = torch.empty((B, H, T, 1), **f32)
        with _lib.on_device(qkvb):
            rc = _lib.lib().fwp_deltanet_prep_fwd(qkvb.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                                                  beta.data_ptr(), T, B, H, D, float(q_scale),
                                                  _lib.stream_of(qkvb))
        _lib.check(rc, "fwp_deltanet_prep_fwd")
        ctx.save_for_backward(qkvb)
        ctx.dims = (T, B, H, D, float(q_scale))
        return q, k, v, beta

    @staticmethod
    def backward(ctx, gq, gk, gv, gbeta):
        (qkvb,) = ctx.saved_tensors
        T, B, H, D, q_scale = ctx.dims
        gq, gk, gv, gbeta = (g.contiguous() for g in (gq, gk, gv, gbeta))
        gqkvb = torch.empty_like(qkvb)
        with _lib.on_device(qkvb):
            rc = _lib.lib().fwp_deltanet_prep_bwd(qkvb.data_ptr(), gq.data_ptr(), gk.data_ptr(), gv.data_ptr(),
                                                  gbeta.data_ptr(), gqkvb.data_ptr(), T, B, H, D, q_scale,
                                                  _lib.stream_of(qkvb))
        _lib.check(rc, "fwp_deltanet_prep_bwd")
        return gqkvb, None, None, None


class DeltaNetLayer(nn.Module):
    """Delta-rule linear-Transformer layer (the reference's
    ``CudaFastWeightLinearTransformerLayer`` with its default
    ``skip_attn_normalization=True``).

    ``h`` is ``[len, bsz, d_model]``.  One projection gives q, k, v and a scalar
    write strength per head; q and k go through :func:`sum_normalised_elu`, beta
    through a sigmoid, and the fast weight memory ``W[bsz, n_head, D, D]`` (zero, or
    ``mems[0]`` when a segment's state is carried over) is updated step by step by
    ``fast_weight_delta``.  The read-out is scaled by ``1/sqrt(D)``, projected, and
    added to the input with LayerNorm.  With ``carry_over_fast_weight`` the call
    returns ``(output, (W_final, None))``.
    """

    def __init__(self, n_head, d_model, d_head, dropout=0.0, dropatt=0.0, pre_lnorm=False,
                 layer_id=None, num_layer=None, fast_weight_op=None):
        super().__init__()
        self.n_head, self.d_model, self.d_head, self.dropout = n_head, d_model, d_head, dropout
        self.layer_id, self.num_layer = layer_id, num_layer
        self.qkvb_net = nn.Linear(d_model, n_head * (3 * d_head + 1), bias=False)
        self.drop = nn.Dropout(dropout)
        self.dropatt = nn.Dropout(dropatt)
        self.o_net = nn.Linear(n_head * d_head, d_model, bias=False)
        self.layer_norm = nn.LayerNorm(d_model)
        self.scale = 1.0 / d_head ** 0.5
        self.pre_lnorm = pre_lnorm
        self.fast_weight_op = fast_weight_op or fast_weight_delta

    def _state(self, mems, carry_over_fast_weight, bsz, h, dtype):
        """The state the operator starts from and overwrites: zeros, or a copy of what was carried over."""
        if mems is None:
            return torch.zeros(bsz, self.n_head, self.d_head, self.d_head, device=h.device, dtype=dtype)
        if not carry_over_fast_weight:
            raise ValueError("mems are only meaningful with carry_over_fast_weight=True")
        # the last batch of an epoch may be smaller than the carried state
        return mems[0][:bsz].clone()

    def forward(self, h, attn_mask=None, mems=None, carry_over_fast_weight=False):
        slen, bsz, _ = h.shape
        H, D = self.n_head, self.d_head
        x = _layer_norm(self.layer_norm, h) if self.pre_lnorm else h
        # The reference's pre-LN branch adds the normalised input back (it rebinds h, :100-104).
        residual = x

        hip_op = self.fast_weight_op is fast_weight_delta
        blocks = None
        if (hip_op and _untouched(self.qkvb_net, nn.Linear) and _untouched(self.o_net, nn.Linear)
                and self.qkvb_net.bias is None and self.o_net.bias is None and _untouched(self.drop, nn.Dropout)):
            blocks = _blocks("takes_delta_block", x, self.qkvb_net.weight, self.o_net.weight, H, D)
        if blocks is not None:
            # the block fills a state that starts at zero itself, beside its pre-step
            fresh = mems is None and getattr(self._state, "__func__", None) is _zeros_or_carried
            W = (torch.empty(bsz, H, D, D, device=h.device, dtype=torch.float32) if fresh
                 else self._state(mems, carry_over_fast_weight, bsz, h, torch.float32))
            drops = _drops(self.drop)
            out = blocks.delta_block(x, self.qkvb_net.weight, self.o_net.weight, W, H, D, self.scale, not drops, fresh)
            if drops:
                out = residual + self.drop(out)
            if not self.pre_lnorm:
                out = _layer_norm(self.layer_norm, out)
            return (out, (W.detach(), None)) if carry_over_fast_weight else out

        qkvb = self.qkvb_net(x)
        fused = hip_op and DeltaNetPrep.supported(qkvb, D)
        if fused:
            # one fused kernel each way; q carries the 1/sqrt(D) of the read-out (the operator is
            # linear in q), and the operator writes [len, bsz, H, D] storage: no pass over its output
            q, k, v, beta = DeltaNetPrep.apply(qkvb, H, D, self.scale)
        else:
            qkvb = qkvb.view(slen, bsz, H, 3 * D + 1)
            q, k, v, beta = (t.permute(1, 2, 0, 3) for t in qkvb.split((D, D, D, 1), dim=-1))
            q, k, beta = sum_normalised_elu(q), sum_normalised_elu(k), torch.sigmoid(beta)

        if hip_op:
            # half or bf16 activations (autocast, which makes some of them fp32): the operator and its state are fp32, as
            # the reference's kernel and its torch.zeros state are
            q, k, v, beta = q.float(), k.float(), v.float(), beta.float()
        W = self._state(mems, carry_over_fast_weight, bsz, h, torch.float32 if hip_op else q.dtype)

        if fused:
            out = fast_weight_delta(q, k, v, beta, W, True)          # [bsz, H, slen, D] over [slen, bsz, H, D] storage
            out = out.permute(2, 0, 1, 3).reshape(slen, bsz, H * D)  # a view
        else:
            out = self.fast_weight_op(q, k, v, beta, W)              # [bsz, H, slen, D]
            out = (self.scale * out).permute(2, 0, 1, 3).reshape(slen, bsz, H * D).to(x.dtype)
        out = residual + self.drop(self.o_net(out))
        if not self.pre_lnorm:
            out = self.layer_norm(out)
        if carry_over_fast_weight:
            return out, (W.detach(), None)
        return out


_zeros_or_carried = DeltaNetLayer._state      # as it is here, whatever replaces it later


class DeltaNetDecoderLayer(nn.Module):
    """Delta-Net layer followed by the feed-forward block (``DecoderLayer`` with
    ``attn_type=24``, model_main.py:703-775); sub-module names ``dec_attn`` and
    ``pos_ff`` as there."""

    def __init__(self, n_head, d_model, d_head, d_inner, dropout=0.0, dropatt=0.0, pre_lnorm=False,
                 layer_id=None, num_layer=None, fast_weight_op=None):
        super().__init__()
        self.dec_attn = DeltaNetLayer(n_head, d_model, d_head, dropout, dropatt, pre_lnorm,
                                      layer_id, num_layer, fast_weight_op)
        self.pos_ff = PositionwiseFF(d_model, d_inner, dropout, pre_lnorm)

    def forward(self, dec_inp, dec_attn_mask=None, mems=None, carry_over_fast_weight=False):
        out = self.dec_attn(dec_inp, attn_mask=dec_attn_mask, mems=mems,
                            carry_over_fast_weight=carry_over_fast_weight)
        if carry_over_fast_weight:
            out, new_mem = out
            return self.pos_ff(out), new_mem
        return self.pos_ff(out)
