"""Layer wrapper WinogradConv, after ResNet-18-var/winograd_conv.py:15-28."""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import swc_hip  # noqa: E402
import winograd2x2_conv.winograd2x2_conv  # noqa: E402

_native = swc_hip.native()

__all__ = ["WinogradConv"]


class WinogradConv(torch.nn.Module):
    """Holds the Winograd-domain weights W [16, in_channel, out_channel] and applies the op.

    Arguments follow ``WinogradConv(x, in_channel, out_channel, mask=None, W_init=None)``
    of the reference (winograd_conv.py:16), with ``x`` moved to ``forward``:

    * ``W_init``: callable filling a tensor in place, or a tensor/array of the weight's
      shape.  Default: the reference's ``variance_scaling_initializer(factor=2*9/32)``
      (:18-19): a normal truncated at two standard deviations with
      std = sqrt(1.3*factor/fan_in), fan_in = 16*in_channel as TensorFlow 1.x computes
      it for a rank-3 shape.
    * ``mask``: optional 0/1 array of the weight's shape; the reference multiplies it in on
      every step (:23-25).  Here W*mask is recomputed only while gradients are being recorded
      (so that they flow to W through the mask); otherwise the product is cached until W or
      mask is written to again (in place or replaced).

    W is a trainable parameter; gradients come from ``winograd2x2_conv_grad``.
    """

    _pieces = None   # also for a layer that was pickled without it

    def __init__(self, in_channel, out_channel, mask=None, W_init=None, precision="fp32", device=None):
        super().__init__()
        self.in_channel, self.out_channel, self.precision = int(in_channel), int(out_channel), precision
        W = torch.empty(16, self.in_channel, self.out_channel, dtype=torch.float32, device=device)
        if W_init is None:
            std = math.sqrt(1.3 * (2.0 * 9.0 / 32.0) / (16 * self.in_channel))
            torch.nn.init.trunc_normal_(W, mean=0.0, std=std, a=-2 * std, b=2 * std)
        elif callable(W_init):
            W_init(W)
        else:
            W.copy_(torch.as_tensor(W_init, dtype=torch.float32).reshape(W.shape))
        self.W = torch.nn.Parameter(W)
        if mask is not None:
            mask = torch.as_tensor(mask, dtype=torch.float32, device=W.device).reshape(W.shape).clone()
        self.register_buffer("mask", mask)
        self._masked = None
        self._bf16 = None

    def __getstate__(self):
        return dict(self.__dict__, _masked=None, _bf16=None, _pieces=None)   # made anew by the copy

    def __setstate__(self, state):
        super().__setstate__(dict(state, _masked=None, _bf16=None, _pieces=None))   # also for a state that holds them in another form

    def refresh(self):
        """Drop the cached W*mask, its bf16 copy and its pieces.  Not needed after in-place updates of W or mask made on
        the tensors themselves or on ``detach()``ed views of them (optimizer steps, ``load_state_dict``,
        ``with torch.no_grad(): W.mul_(m)``): the caches are keyed on the tensors' version counters and storage,
        so those are noticed by themselves.  Needed after a write through ``.data`` (``layer.W.data.mul_(m)``,
        ``layer.W.data.copy_(w)``): a ``.data`` view carries a version counter of its own, so such a write leaves
        no trace on W."""
        self._masked = None
        self._bf16 = None
        self._pieces = None

    def _weight_key(self):
        # In-place writes bump _version; a replaced or moved tensor changes data_ptr / device.
        return _native.key(self.W, self.mask)

    def _keep(self, slot, key, tensor, *made_for):
        """``tensor``, made of the weights that ``key`` stands for, kept in ``slot`` with a mark behind it in the stream that wrote it: a
        call on another stream may find it before it has been written, or drop it (the weights changed) while that stream's kernels
        read it, and ``kept`` sees to both.  While a graph is captured nothing is kept: what the capture records is written when the
        graph runs, and other calls would read it before."""
        mark = _native.mark(tensor)
        if mark is not None:
            setattr(self, slot, (key, tensor, mark) + made_for)
        return tensor

    def bf16_weight(self):
        """W*mask as the [16,K,C] bfloat16 tensor the bf16-stored kernel reads; cached like masked_weight()."""
        tensor = _native.kept(self._bf16, self.W, self.mask)
        if tensor is not None:
            return tensor
        return self._keep("_bf16", self._weight_key(), winograd2x2_conv.winograd2x2_conv.winograd2x2_weights_bf16(self.masked_weight()))

    def weight_pieces(self):
        """W*mask taken apart for the fp32 convolution, or rounded and put in order for the one with bf16 operands; cached like masked_weight()."""
        return self._pieces_of(self.masked_weight())

    def _pieces_of(self, masked):
        precision, entry = self.precision, self._pieces
        tensor = _native.kept(entry, self.W, self.mask) if entry is not None and entry[3] == precision else None
        if tensor is not None:
            return tensor
        key = self._weight_key()
        if self.mask is not None:   # the key that `masked` was made under: another thread may have written to W since
            source = self._masked
            key = source[0] if source is not None and source[1] is masked else None
        pieces = winograd2x2_conv.winograd2x2_conv.winograd2x2_weight_pieces(masked, precision)
        return self._keep("_pieces", key, pieces, precision) if key is not None else pieces

    def masked_weight(self):
        """W*mask without autograd history, recomputed only when W or mask changed since the last call (a write
        through ``.data`` is not such a change: see refresh())."""
        W, mask = self.W, self.mask
        if mask is None:
            return W.detach()   # shares W's version counter: a write to what is handed out is noticed
        tensor = _native.kept(self._masked, W, mask)
        if tensor is not None:
            return tensor
        return self._keep("_masked", _native.key(W, mask), (W.detach() * mask).contiguous())

    def forward(self, x, affine=None, residual=None, residual_relu=False):
        """``affine=(scale, shift)`` and ``residual`` (forward only) are applied to the result inside
        the kernel: ``conv*scale + shift + residual`` (``+ relu(residual)`` with ``residual_relu``)."""
        pieces = None
        if x.dtype == torch.bfloat16:      # bf16-stored activations: forward only
            w = self.bf16_weight()
        elif torch.is_grad_enabled() and self.W.requires_grad:
            w = self.W if self.mask is None else self.W * self.mask
            pieces = True
        else:
            w = self.masked_weight()
            # the cached pieces where W*mask is cached too, pieces made for this call where W itself is used
            if self.mask is None:
                pieces = True
            elif self.precision in ("fp32", "bf16"):
                if _native.pieces_gain(x, self.out_channel, self.precision == "bf16") and x.device == w.device and x.shape[4] == w.shape[1]:
                    pieces = self._pieces_of(w)
        scale, shift = affine if affine is not None else (None, None)
        return winograd2x2_conv.winograd2x2_conv.winograd2x2_conv(x, w, self.precision, None, scale, shift, residual, residual_relu, True, pieces)
