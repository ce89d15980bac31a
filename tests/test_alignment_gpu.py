"""Tensors at addresses that are no multiple of 16: parameters that are slices of a flat buffer, saved tensors that hooks
restore elsewhere, buffers of a C caller.  What the wide kernels cannot take runs through others, with the same results."""
import ctypes

import pytest
import torch

from tests.helpers import assert_close

pytestmark = pytest.mark.gpu
SEED = 0xC0FFEE


def _odd(t):
    """t's values two bytes past a multiple of 16."""
    return torch.empty(t.numel() + 8, dtype=t.dtype, device='cuda')[1:1 + t.numel()].view(t.shape).copy_(t)


def _encoder(dims, act, which='mi355x', **more):
    from substation_amd import Encoder, layouts as L
    lay = L.mi355x_layouts() if which == 'mi355x' else L.reference_layouts(which)
    torch.manual_seed(0)
    B, Ls, H, E = dims
    enc = Encoder('unused', B, Ls, H, E, lay, torch.float16, 0.1, 0.1, 0.1, 0.1, activation=act, seed=SEED, **more).cuda()
    with torch.no_grad():
        for q in enc.parameters():
            q.mul_(0.1)
    g = torch.Generator().manual_seed(5)
    x, dy = (torch.randn([enc.sizes[d] for d in lay[k][1]], generator=g).half().cuda() for k in ('input', 'output'))
    return enc, x.requires_grad_(), dy


def _pass(enc, x, dy, call=None, hooks=None):
    x.grad = None
    enc.zero_grad(set_to_none=True)
    enc.set_rng(SEED, 0)
    with hooks or torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        y = (call or enc)(x)
    y.backward(dy)
    return dict([('SB2', y.detach()), ('DX', x.grad)] + [('D' + n, q.grad) for n, q in enc.named_parameters()])


def _c_pass(enc, x, dy, odd, between=lambda: None):
    """Both passes as a C caller makes them, with the named buffers (parameters, intermediates, 'D' + parameter) at odd
    addresses; intermediates start as NaN."""
    handle, lay = enc._handle, enc.layouts
    handle.set_stream(torch.cuda.current_stream().cuda_stream)
    place = lambda n, t: _odd(t) if n in odd else t

    def call(name, args):
        from substation_amd import _lib
        ptrs = (ctypes.c_void_p * len(args))(*(t.data_ptr() for t in args))
        _lib.check(getattr(handle.lib, 'sub_encoder_' + name)(handle.ptr, ptrs, len(args)), name)
    params = [place(n, getattr(enc, n).detach()) for n, _ in lay['params']]
    grads = [place('D' + n, torch.full_like(q, float('nan'))) for (n, _), q in zip(lay['params'], params)]
    fwd, bwd = ([place(n, torch.full([enc.sizes[d] for d in o], float('nan'), dtype=torch.float16, device='cuda'))
                 for n, o in lay[k]] for k in ('forward_interm', 'backward_interm'))
    y, dx = torch.empty_like(dy), torch.empty_like(x)
    enc.set_rng(SEED, 0)
    call('forward', [x, *params, *fwd, y])
    between()
    call('backward', [dy, *grads, *bwd, *params, *fwd, x, dx])
    return dict([('SB2', y), ('DX', dx)] + [('D' + n, t) for (n, _), t in zip(lay['params'], grads)])


def _close(got, want):
    # values rounded to fp16 between operators, the products' terms added in another order: the bound of the layer's tests
    for n, t in want.items():
        assert_close(got[n].float().cpu().numpy(), t.float().cpu().numpy(), name=n)


@pytest.mark.parametrize('dims', [(2, 128, 12, 768), (2, 40, 2, 128), (8, 512, 8, 512)])
@pytest.mark.parametrize('odd', [('LINW2',), ('DLIN1',), ('DLIN2',), ('LINW2', 'DLIN1', 'DLIN2')])
def test_gelu_layer_whose_backward_epilogue_finds_a_misaligned_tensor(dims, odd):
    """The forward epilogue leaves the keep bits and no mask; the backward operator takes them where the backward epilogue
    cannot run: B=8 L=512 has whole 256 x 256 tiles, the others have not."""
    enc, x, dy = _encoder(dims, 'gelu')
    want = _pass(enc, x, dy)
    _close(_c_pass(enc, x.detach(), dy, odd), want)
    if odd == ('LINW2',):
        enc.LINW2.data = _odd(enc.LINW2.data)
        _close(_pass(enc, x, dy), want)


def test_decoder_layer_whose_parameters_are_misaligned():
    """2048 x 4096 feed-forward outputs: 128 tiles of 256 x 256, so linear1 carries its activation.  The second feed-forward
    weight at an odd address in both passes; every parameter restored to one for the backward pass."""
    from substation_amd import DecoderLayer
    torch.manual_seed(0)
    layer = DecoderLayer(8, 256, 128, 4, 256, 0.1, 0.1, 0.1, 0.1, activation='gelu', seed=SEED, intermediate_size=4096).cuda()
    x, src, dy = (torch.randn(8, n, 256).half().cuda() for n in (256, 128, 256))

    def both_passes(restore=lambda t: t):
        layer.zero_grad(set_to_none=True)
        layer.set_rng(SEED, 1)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, restore):
            y = layer(x, src)
        assert layer.ffn_in_epilogues
        y.backward(dy)
        return dict([('y', y.detach())] + [(n, q.grad) for n, q in layer.named_parameters()])
    want = both_passes()
    _close(both_passes(_odd), want)
    layer.linear2_w.data = _odd(layer.linear2_w.data)
    _close(both_passes(), want)


@pytest.mark.parametrize('act', ['relu', 'gelu'])
@pytest.mark.parametrize('python', [False, True])
@pytest.mark.parametrize('persistent', [False, True])
@pytest.mark.parametrize('what', ['LINW1', 'all', 'strided'])
def test_saved_tensors_that_hooks_restore_elsewhere(act, python, persistent, what):
    """Restored to addresses that are no multiple of 16, or with other strides: the backward pass takes what its forward pass
    left for it, bit for bit as without hooks (at 2 x 128 x 768 the two passes run with activation epilogues)."""
    enc, x, dy = _encoder((2, 128, 12, 768), act, persistent_workspace=persistent)
    call = (lambda t: enc.encoder_func.apply(t, *enc.params)) if python else enc
    want = {n: t.clone() for n, t in _pass(enc, x, dy, call).items()}

    def restore(t):
        if what == 'strided':
            return t.t().contiguous().t() if t.dim() == 2 else t
        return _odd(t) if what == 'all' or t.shape == enc.LINW1.shape else t
    got = _pass(enc, x, dy, call, torch.autograd.graph.saved_tensors_hooks(lambda t: t, restore))
    for n, t in want.items():
        assert torch.equal(got[n], t), n


@pytest.mark.parametrize('act', ['relu', 'gelu'])
@pytest.mark.parametrize('python', [False, True])
def test_saved_tensors_restored_aligned_that_were_not(act, python):
    """The other way round: the forward pass finds LINW1 misaligned and runs bias, activation and dropout as an operator; a
    hook restores it aligned."""
    enc, x, dy = _encoder((2, 128, 12, 768), act)
    call = (lambda t: enc.encoder_func.apply(t, *enc.params)) if python else enc
    enc.LINW1.data = _odd(enc.LINW1.data)
    assert enc.LINW1.data_ptr() % 16
    want = _pass(enc, x, dy, call)
    _close(_pass(enc, x, dy, call, torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.clone())), want)


def test_backward_call_that_cannot_take_what_its_forward_call_left_refuses():
    """A C caller says what its forward call left; without attention in registers (switched off in between, which is also
    what a tensor at an odd address does) there is no backward pass for that, and none is begun."""
    from substation_amd import _lib
    enc, x, dy = _encoder((2, 128, 2, 128), 'gelu')
    form = ctypes.c_int(-1)

    def say():
        _lib.check(enc._handle.lib.sub_forward_form(enc._handle.ptr, ctypes.byref(form)))
        _lib.check(enc._handle.lib.sub_set_forward_form(enc._handle.ptr, form))
    want = _c_pass(enc, x.detach(), dy, ())
    got = _c_pass(enc, x.detach(), dy, (), say)
    assert form.value > 0
    with pytest.raises(_lib.SubstationError):
        _c_pass(enc, x.detach(), dy, (), lambda: (say(), enc._handle.set_option(4, 0)))
    _c_pass(enc, x.detach(), dy, ())              # said for that one call only
    for n, t in want.items():
        assert torch.equal(got[n], t), n


@pytest.mark.parametrize('odd', [('LINW1',), ('LINW2',), ('LINW1', 'LINW2', 'DLINW1', 'DLINW2')])
@pytest.mark.parametrize('act', ['relu', 'gelu'])
def test_misaligned_feed_forward_weights_of_feature_major_layouts(odd, act):
    """Under a configuration that the layer runs in its own orders, LINW1 and LINW2 are read and written as they lie; where
    they lie misaligned, by way of copies, like the other weights: the launches and the bits are those of aligned ones."""
    enc, x, dy = _encoder((2, 128, 12, 768), act, 'bert-b8-l512-h16-e1024')
    enc._handle.profile_enable(True)
    want = _c_pass(enc, x.detach(), dy, ())
    launches = [n for n, _ in enc._handle.profile_read()]
    got = _c_pass(enc, x.detach(), dy, odd)
    assert [n for n, _ in enc._handle.profile_read()] == launches and 'lin1+bad' in launches and 'dXlin2+bdrlb' in launches
    for n, t in want.items():
        assert torch.equal(got[n], t), n
    # and with saved tensors and other addresses in every pass
    for n in ('LINW1', 'LINW2'):
        if n in odd:
            getattr(enc, n).data = _odd(getattr(enc, n).data)
    for n, t in _pass(enc, x, dy).items():
        assert torch.equal(want[n], t), n


@pytest.mark.parametrize('python', [False, True])
@pytest.mark.parametrize('restore', [lambda t: t.cpu(), lambda t: t.float(), lambda t: t.reshape(-1)[:8]])
def test_saved_tensors_that_hooks_restore_as_something_else_are_refused(python, restore):
    """On another device, with another type or size: an error in front of the first launch, not bare pointers to it."""
    enc, x, dy = _encoder((2, 128, 2, 128), 'gelu')
    call = (lambda t: enc.encoder_func.apply(t, *enc.params)) if python else enc
    want = _pass(enc, x, dy, call)
    with pytest.raises(RuntimeError, match='restored'):
        _pass(enc, x, dy, call, torch.autograd.graph.saved_tensors_hooks(lambda t: t, restore))
    for n, t in _pass(enc, x, dy, call, torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t.reshape(-1))).items():
        assert torch.equal(want[n], t.reshape(want[n].shape)), n
