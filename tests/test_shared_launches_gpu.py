"""Launches of several products: tiles of up to seven of them in one schedule, against the products launched one by one."""
import pytest
import torch

from tests.helpers import assert_close

pytestmark = pytest.mark.gpu

ALL = 'dXQKV-fused+dWQKV-fused+dWout+dWlin1+dWlin2'


# (B, L, H, E), layouts, a launch that has to be among them (None: whichever)
CASES = [
    ((1, 16, 2, 128), None, None),                   # fewer tiles than one product's
    ((3, 43, 4, 256), None, None),                   # rows that are a multiple of nothing
    ((5, 201, 12, 768), None, None),                 # remainders of every tile size
    ((4, 512, 16, 1024), None, ALL),
    ((8, 512, 16, 1024), None, ALL),                 # 256 x 256 tiles, a round of them exactly
    ((48, 128, 16, 1024), 'bert-b96-l128-h16-e1024', ALL),     # data gradients with both operands along k
    ((2, 1024, 32, 2048), None, None),               # several rounds
    ((1, 2048, 32, 4096), None, None),               # whole rounds in front of the parts of the schedule
]


@pytest.mark.parametrize('dims,which,launch', CASES)
def test_products_that_share_a_launch_give_what_they_give_alone(dims, which, launch):
    from substation_amd import Encoder, layouts as L
    B, Ls, H, E = dims
    lay = L.mi355x_layouts(which)
    g = torch.Generator('cuda').manual_seed(3)
    sizes = L.sizes_map(B, Ls, H, E)
    X, DY = (torch.randn(L.shape_of(lay[k][1], sizes), generator=g, device='cuda').half() for k in ('input', 'output'))
    grads = []
    for shared in (0, 1):
        torch.manual_seed(0)
        with torch.device('cuda'):
            enc = Encoder('unused', B, Ls, H, E, lay, torch.float16, 0.1, 0.1, 0.1, 0.1, seed=7, activation='gelu', profiling=True)
        with torch.no_grad():
            for q in enc.parameters():
                q.mul_(0.1)
        enc._handle.set_option(5, shared)
        enc.set_rng(7, 0)
        x = X.clone().requires_grad_()
        enc(x).backward(DY)
        torch.cuda.synchronize()
        names = [n for n, _ in enc.profile()]
        assert shared or not any('+dW' in n for n in names)
        assert not (shared and launch) or launch in names, names
        grads.append({'X': x.grad, **{n: q.grad for n, q in enc.named_parameters()}})
    for name, alone in grads[0].items():
        # (sums in another order, rounded to fp16, and what follows from them: within the bound of any product here)
        assert_close(grads[1][name].float().cpu().numpy(), alone.float().cpu().numpy(), tol=1e-2, name=name)


@pytest.mark.parametrize('dims,source', [((2, 128, 2, 128), 256), ((3, 40, 4, 256), 72), ((4, 384, 16, 1024), 128)])
def test_group_of_contractions_gives_what_each_of_them_gives(dims, source):
    """Ten products of two sizes in one call, one of them added to its own output, against single calls."""
    from substation_amd.ops import Ops
    B, Ls, H, E = dims
    o, os_ = Ops(B, Ls, H, E), Ops(B, source, H, E)
    g = torch.Generator('cuda').manual_seed(1)

    def tensor(ops, layout):
        return (0.3 * torch.randn(ops.empty(layout).shape, generator=g, device='cuda')).half()

    products, alone = [], []
    for ops, la, lb, lc, lt in [(o, 'QHPI', 'QBJHP', 'BJI', 'BJI'), (os_, 'BKHP', 'HPI', 'BKI', 'BKI'), (os_, 'BKHP', 'BKI', 'HPI', None),
                                (os_, 'BKHP', 'BKI', 'HPI', None), (o, 'QBJHP', 'BJI', 'QHPI', None), (o, 'BJI', 'BJHP', 'IHP', None),
                                (o, 'BJHP', 'BJI', 'HPI', None), (o, 'BJI', 'BJHP', 'IHP', None), (o, 'BJU', 'BJI', 'UI', None),
                                (o, 'BJI', 'BJU', 'IU', None)]:
        a, b, c = tensor(ops, la), tensor(ops, lb), tensor(ops, lc)
        want = ops.empty(lc)
        if lt:
            ops.einsum(a, la, b, lb, want, lc, addend=c, l_addend=lt)
            products.append((ops, a, la, b, lb, c, lc, c, lt))
        else:
            ops.einsum(a, la, b, lb, want, lc)
            products.append((ops, a, la, b, lb, c, lc))
        alone.append(want)
    o.einsum_group(products)
    for (_, _, la, _, lb, c, lc, *_), want in zip(products, alone):
        # fp32 sums in another order, rounded once
        assert_close(c.float().cpu().numpy(), want.float().cpu().numpy(), tol=2e-3, name=f'{la},{lb}->{lc}')


@pytest.mark.parametrize('dims', [(8, 500, 16, 1024), (5, 43, 4, 256)])
def test_products_after_a_change_of_dimension_orders(dims):
    """Gradients of a layer whose tensors are no longer kept in the library's own orders (option 11) after a pass in them, against one
    that never was in them: tokens contiguous in the feed-forward block, 4000 of them, which is no multiple of 64, and 215."""
    from substation_amd import Encoder, layouts as L
    B, Ls, H, E = dims
    lay = dict(L.mi355x_layouts())
    other = dict(DLIN1='UBJ', DROP2='UBJ', LIN1='UBJ', SB1='IBJ', DLIN2='IBJ', WKQV='QIHP')
    for group in ('params', 'forward_interm', 'backward_interm'):
        lay[group] = [(name, other.get(name, order)) for name, order in lay[group]]
    g = torch.Generator('cuda').manual_seed(3)
    X, DY = (torch.randn(B, Ls, E, generator=g, device='cuda').half() for _ in range(2))
    grads = []
    for before in (False, True):
        torch.manual_seed(0)
        with torch.device('cuda'):
            enc = Encoder('unused', B, Ls, H, E, lay, torch.float16, 0.1, 0.1, 0.1, 0.1, seed=7, activation='gelu')
        with torch.no_grad():
            for q in enc.parameters():
                q.mul_(0.1)
        if before:
            enc(X.clone().requires_grad_()).backward(DY)
            enc.zero_grad(set_to_none=True)
        enc._handle.set_option(11, 0)
        enc.set_rng(7, 0)
        x = X.clone().requires_grad_()
        enc(x).backward(DY)
        grads.append([x.grad] + [q.grad for q in enc.parameters()])
    for a, b in zip(*grads):
        assert torch.equal(a, b)
