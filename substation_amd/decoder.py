"""Decoder layer with encoder-decoder attention on the MI355X operators.

The reference states this layer in NumPy only (``decoder_with_encoder_attention``
and its backward pass, substation/transformer.py:288-441; its CUDA module covers
the encoder layer alone).  Here it runs on the device as a sequence of the
library's operators, issued by the extension module (csrc/host.cpp) -- the contraction kernel with bias and residual addends in
its epilogue, the attention kernels that keep the scores in registers (with an
additive mask for the self-attention and with a key length of their own for the
attention over the encoder output), bdrln / bad and the LayerNorm-backward
operator -- in the order of the reference's statements.

Argument and parameter names follow the reference's (``sattn_*``, ``edattn_*``,
``norm{1,2,3}_*``, ``linear{1,2}_*``).  The three self-attention projections are
one stacked weight, as in the encoder module (index 0 = K, 1 = Q, 2 = V,
pytorch_module/encoder.cu:93-99).  Dropout follows the device contract of the
encoder module: {0,1} masks from the seeded Philox streams, ``y = x * mask``
without rescaling; as in the reference there is none on the attention
probabilities of this layer.
"""
import math
from operator import index

import torch

from . import _lib
from .encoder import causal_mask
from .ops import Ops

#: dropout sites (Philox stream ids) of the four masks, in the order of the constructor's probabilities
SITE_SATTN, SITE_EDATTN, SITE_LINEAR1, SITE_FF = 1, 4, 2, 3


class DecoderLayer(torch.nn.Module):
    """``forward(x, encoder_out)``: x [B, target_len, E], encoder_out [B, source_len, E],
    fp16 on the GPU; returns [B, target_len, E].  Sequence lengths must be
    multiples of 128 and the head size 64 or 128 (the attention kernels' tiles)."""

    def __init__(self, batch_size, target_len, source_len, num_heads, embedding_size,
                 sattn_dropout_p=0.1, edattn_dropout_p=0.1, linear1_dropout_p=0.1, ff_dropout_p=0.1,
                 activation='gelu', seed=0, intermediate_size=None, sattn_mask='causal'):
        super().__init__()
        B, Lt, Ls, H, E = batch_size, target_len, source_len, num_heads, embedding_size
        if E % H:
            raise ValueError('embedding_size must be a multiple of num_heads')
        P, U = E // H, intermediate_size or 4 * E
        if Lt % 128 or Ls % 128 or P not in (64, 128):
            raise ValueError('DecoderLayer: sequence lengths must be multiples of 128 and the head size 64 or 128')
        self.batch_size, self.target_len, self.source_len = B, Lt, Ls
        self.num_heads, self.embedding_size, self.proj_size, self.intermediate_size = H, E, P, U
        self.probs = (sattn_dropout_p, edattn_dropout_p, linear1_dropout_p, ff_dropout_p)
        self.activation = activation
        self.seed, self.step = seed, 0
        self.activation_epilogues = True     # linear1 / its backward with the activation in their epilogues where they qualify
        self.ffn_in_epilogues = False        # whether the last forward call took them
        self.ops_t = Ops(B, Lt, H, E, activation=activation, seed=seed, intermediate_size=U)   # target-side sizes
        self.ops_s = Ops(B, Ls, H, E, activation=activation, seed=seed, intermediate_size=U)   # source-side sizes

        def param(*shape, std=None, fill=None):
            t = torch.empty(shape, dtype=torch.float16)
            if fill is not None:
                t.fill_(fill)
            else:
                t.normal_(0.0, std)
            return torch.nn.Parameter(t)

        w = 1.0 / math.sqrt(E)
        self.sattn_wkqv = param(3, H, P, E, std=w)      # [Q,H,P,I], Q: 0 = K, 1 = Q, 2 = V
        self.sattn_in_b = param(3, H, P, fill=0.0)
        self.sattn_wo = param(E, H, P, std=w)
        self.sattn_out_b = param(E, fill=0.0)
        self.edattn_wq = param(H, P, E, std=w)
        self.edattn_wk = param(H, P, E, std=w)
        self.edattn_wv = param(H, P, E, std=w)
        self.edattn_in_b = param(3, H, P, fill=0.0)     # (q, k, v) order, as the reference's in_b
        self.edattn_wo = param(E, H, P, std=w)
        self.edattn_out_b = param(E, fill=0.0)
        for i in (1, 2, 3):
            setattr(self, f'norm{i}_scale', param(E, fill=1.0))
            setattr(self, f'norm{i}_bias', param(E, fill=0.0))
        self.linear1_w = param(U, E, std=w)
        self.linear1_b = param(U, fill=0.0)
        self.linear2_w = param(E, U, std=1.0 / math.sqrt(U))
        self.linear2_b = param(E, fill=0.0)
        self.param_names = [n for n, _ in self.named_parameters()]
        if isinstance(sattn_mask, str):
            if sattn_mask != 'causal':
                raise ValueError("sattn_mask: 'causal', None or an additive [target_len, target_len] tensor")
            sattn_mask = causal_mask(Lt, 'cpu')
        self.register_buffer('sattn_mask', sattn_mask, persistent=False)
        self._function = _make_function(self)

    def set_rng(self, seed, step=0):
        """The four masks of forward call number ``step`` are functions of (seed, step) only."""
        self.seed, self.step = seed, step

    def forward(self, x, encoder_out):
        return self._function.apply(x, encoder_out, *[getattr(self, n) for n in self.param_names])


def _make_function(m):
    o, os_ = m.ops_t, m.ops_s
    scale = 1.0 / math.sqrt(m.proj_size)
    # the operators of both passes (host.cpp, DecoderPasses): parameters in the order in which they are registered above
    Passes = _lib.host().DecoderPasses            # (and its places in what a forward pass returns)
    passes = Passes(
        o.handle.ptr, os_.handle.ptr, (o, os_),
        [m.batch_size, m.target_len, m.source_len, m.num_heads, m.proj_size, m.embedding_size, m.intermediate_size],
        [float(p) for p in m.probs], [SITE_SATTN, SITE_EDATTN, SITE_LINEAR1, SITE_FF], m.activation == 'relu', scale)

    class DecoderFunction(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x, enc, *params):
            if not (x.is_cuda and enc.is_cuda):
                raise RuntimeError('DecoderLayer.forward needs tensors on the GPU')
            x, enc = x.contiguous(), enc.contiguous()
            step, m.step = m.step, m.step + 1
            ctx.mask = m.sattn_mask
            kept = passes.forward(x, enc, params, ctx.mask, index(m.seed) & (2**64 - 1), index(step) & (2**32 - 1), bool(m.activation_epilogues))
            y = kept.pop(Passes.OUTPUT)
            m.ffn_in_epilogues = kept[Passes.BITS] is not None
            ctx.save_for_backward(x, enc, *params)
            ctx.kept = kept
            m.last_masks = dict(sattn=kept[Passes.MASK1], edattn=kept[Passes.MASK2], linear1=kept[Passes.MASK3], ff=kept[Passes.MASK4])
            return y

        @staticmethod
        def backward(ctx, dy):
            x, enc, *params = ctx.saved_tensors
            return tuple(passes.backward(x, enc, params, ctx.kept, dy.contiguous(), ctx.mask))

    return DecoderFunction
