"""Forward passes that no backward pass follows (sub_forward_alone): the same output, and nothing kept."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# sizes on each of the tile forms of lin1 with its activation, split lin2 (its sums go into the LayerNorm), and remainders
@pytest.mark.parametrize('act', ['gelu', 'relu'])
@pytest.mark.parametrize('p', [0.0, 0.1])
@pytest.mark.parametrize('dims', [(1, 16, 16, 1024), (1, 64, 12, 768), (3, 43, 4, 256), (24, 77, 12, 768), (13, 201, 12, 768),
                                  (8, 512, 16, 1024), (1, 128, 32, 4096)])
def test_a_forward_pass_without_gradients_gives_the_same_output(dims, p, act):
    from substation_amd import Encoder, layouts as L
    B, Ls, H, E = dims
    torch.manual_seed(0)
    with torch.device('cuda'):
        enc = Encoder('unused', B, Ls, H, E, L.mi355x_layouts(), torch.float16, p, p, p, p, seed=7, activation=act)
        x = torch.randn(B, Ls, E).half()
    with torch.no_grad():
        for q in enc.parameters():
            q.mul_(0.1)
    enc.set_rng(7, 0)
    want = enc(x.clone().requires_grad_()).detach()
    enc.set_rng(7, 0)
    with torch.no_grad():
        got = enc(x)
    assert torch.equal(got, want)


def test_a_backward_pass_belongs_to_the_forward_pass_before_one_without_gradients():
    from substation_amd import Encoder, layouts as L
    torch.manual_seed(0)
    with torch.device('cuda'):
        enc = Encoder('unused', 2, 128, 4, 256, L.mi355x_layouts(), torch.float16, 0.1, 0.1, 0.1, 0.1, seed=7, activation='gelu')
        x, other, dy = (torch.randn(2, 128, 256).half() for _ in range(3))
    grads = []
    for between in (False, True):
        enc.set_rng(7, 0)
        leaf = x.clone().requires_grad_()
        y = enc(leaf)
        if between:
            with torch.no_grad():
                enc(other)
        y.backward(dy)
        grads.append([leaf.grad] + [q.grad for q in enc.parameters()])
        enc.zero_grad(set_to_none=True)
    for a, b in zip(*grads):
        assert torch.equal(a, b)


def test_a_call_that_needs_what_was_not_kept_is_refused():
    from substation_amd import _lib
    from substation_amd import layout_search as ls, layouts as L
    timer = ls.LayerTimer(1, 64, 2, 128, iters=1, warmup=1)
    lay = L.mi355x_layouts()
    lib, handle = _lib.load(), timer._handle(lay, False)
    handle.set_option(12, 1)
    fp, nf, bp, nb = timer._pointers(lay)
    _lib.check(lib.sub_forward_alone(handle.ptr), 'sub_forward_alone')
    _lib.check(lib.sub_encoder_forward(handle.ptr, fp, nf), 'encoder_forward')
    with pytest.raises(RuntimeError, match='sub_forward_alone'):
        _lib.check(lib.sub_encoder_backward(handle.ptr, bp, nb), 'encoder_backward')
    _lib.check(lib.sub_encoder_forward(handle.ptr, fp, nf), 'encoder_forward')
    _lib.check(lib.sub_encoder_backward(handle.ptr, bp, nb), 'encoder_backward')
    torch.cuda.synchronize()
    handle.close()
