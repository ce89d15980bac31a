"""In front of a ReLU the order of a product's sums is a fixed function of its shape."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dims', [(2, 128, 12, 768), (4, 256, 12, 768), (13, 201, 12, 768), (8, 512, 16, 1024), (2, 1024, 16, 2048)])
def test_gates_do_not_depend_on_how_the_activation_is_launched(dims):
    """lin1 with its activation in one launch and operator by operator: the same gates, so the same gradients to rounding, without
    a single element moved by a gate that fell the other way (3 % and more of its row's size)."""
    from substation_amd import Encoder, layouts as L
    B, Ls, H, E = dims
    g = torch.Generator('cuda').manual_seed(5)
    x, dy = (torch.randn(B, Ls, E, generator=g, device='cuda').half() for _ in range(2))
    got = []
    for epilogues in (1, 0):
        torch.manual_seed(0)
        with torch.device('cuda'):
            enc = Encoder('unused', B, Ls, H, E, L.mi355x_layouts(), torch.float16, 0.1, 0.1, 0.1, 0.1, seed=7, activation='relu',
                          profiling=True)
        with torch.no_grad():
            for q in enc.parameters():
                q.mul_(0.3)
        enc._handle.set_option(1, epilogues)
        enc.set_rng(7, 0)
        leaf = x.clone().requires_grad_()
        y = enc(leaf)
        y.backward(dy)
        got.append((y.detach(), enc.LINB1.grad))
        torch.cuda.synchronize()
        assert ('lin1+bad' in [n for n, _ in enc.profile()]) == bool(epilogues)
    assert torch.equal(got[0][0], got[1][0])
    a, b = (t[1].float() for t in got)
    assert float((a - b).abs().max()) <= 4e-3 * float(a.abs().max())
