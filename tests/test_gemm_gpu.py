"""GPU parity of the einsum contraction (MFMA kernel and scalar fallback) against
numpy.einsum in fp64 on the same fp16-rounded operands, for all 18 contractions
of the layer under the MI355X layouts and both layouts the reference ships.
fp16 products accumulate in fp32 and are rounded once: tolerance 1e-2 relative."""
import numpy as np
import pytest
import torch

from tests.einsums import EINSUMS, operand_layouts
from tests.helpers import assert_close, from_layout, h16, to_layout

pytestmark = pytest.mark.gpu


def _layout_sets():
    from substation_amd import layouts as L
    return [('mi355x', L.mi355x_layouts()), ('ref-b8', L.reference_layouts('bert-b8-l512-h16-e1024')),
            ('ref-b96', L.reference_layouts('bert-b96-l128-h16-e1024'))]


@pytest.mark.parametrize('B,L,H,E', [(2, 16, 2, 32), (3, 40, 3, 24), (2, 128, 4, 256), (1, 256, 2, 128)])
def test_all_contractions(B, L, H, E):
    from substation_amd.ops import Ops
    o = Ops(B, L, H, E)
    sz = o.sizes
    rng = np.random.default_rng(7)
    kinds = set()
    for lname, lay in _layout_sets():
        t = operand_layouts(lay)
        for name, a, b, c, scaled in EINSUMS:
            la, lb, lc = t[a], t[b], t[c]
            A = h16(rng.normal(size=tuple(sz[d] for d in la)))
            Bm = h16(rng.normal(size=tuple(sz[d] for d in lb)))
            alpha = 1.0 / np.sqrt(sz['P']) if scaled else 1.0
            want = alpha * np.einsum(f'{la},{lb}->{lc}'.lower(), A, Bm)
            C = torch.full(tuple(sz[d] for d in lc), float('nan'), dtype=torch.float16, device='cuda')
            kinds.add(o.handle.classify(la, lb, lc)['kernel'])
            o.einsum(to_layout(A, la, la), la, to_layout(Bm, lb, lb), lb, C, lc, alpha=alpha)
            torch.cuda.synchronize()
            assert_close(from_layout(C, lc, lc), want, name=f'{lname}:{name} {la},{lb}->{lc}')
    if E % 8 == 0 and L % 8 == 0:
        assert 1 in kinds, 'the MFMA kernel was never selected'


@pytest.mark.parametrize('B,L,H,E', [(2, 67, 2, 128), (1, 129, 1, 40), (3, 5, 2, 6)])
def test_contractions_of_odd_sizes(B, L, H, E):
    """Rows that are not whole 16-byte words: the kernel for any strides and sizes, tiles with remainders on every side."""
    test_all_contractions(B, L, H, E)


def test_k_remainder_and_tile_edges():
    """K not a multiple of the 64-wide LDS tile, M/N not multiples of 128."""
    from substation_amd.ops import Ops
    o = Ops(3, 72, 5, 200)          # P=40, U=800
    sz = o.sizes
    rng = np.random.default_rng(8)
    for la, lb, lc in (('BJI', 'UI', 'BJU'), ('BJU', 'IU', 'BJI'), ('BJI', 'BJU', 'UI'),
                       ('BKHP', 'BJHP', 'BHJK'), ('BHJK', 'BKHP', 'BJHP'), ('BJHP', 'BHJK', 'BKHP')):
        A = h16(rng.normal(size=tuple(sz[d] for d in la)))
        Bm = h16(rng.normal(size=tuple(sz[d] for d in lb)))
        want = np.einsum(f'{la},{lb}->{lc}'.lower(), A, Bm)
        C = torch.full(tuple(sz[d] for d in lc), float('nan'), dtype=torch.float16, device='cuda')
        assert o.handle.classify(la, lb, lc)['kernel'] == 1
        o.einsum(to_layout(A, la, la), la, to_layout(Bm, lb, lb), lb, C, lc)
        torch.cuda.synchronize()
        assert_close(from_layout(C, lc, lc), want, name=f'{la},{lb}->{lc}')


@pytest.mark.parametrize('E,H', [(192, 3), (64, 1), (128, 2)])
def test_wide_tiles_every_operand_orientation(E, H):
    """4096 x 4096 outputs take 256 x 256 tiles: each operand k-contiguous or not, with
    an odd number of 64-deep k-tiles (three, one) and an even one."""
    from substation_amd.ops import Ops
    o = Ops(8, 512, H, E, intermediate_size=4096)
    sz = o.sizes
    rng = np.random.default_rng(E)
    for la in ('BJI', 'IBJ'):
        for lb in ('UI', 'IU'):
            lc = 'BJU'
            A = h16(rng.normal(size=tuple(sz[d] for d in la)))
            Bm = h16(rng.normal(size=tuple(sz[d] for d in lb)))
            want = np.einsum(f'{la},{lb}->{lc}'.lower(), A, Bm)
            C = torch.full(tuple(sz[d] for d in lc), float('nan'), dtype=torch.float16, device='cuda')
            assert o.handle.classify(la, lb, lc)['kernel'] == 1
            o.einsum(to_layout(A, la, la), la, to_layout(Bm, lb, lb), lb, C, lc)
            torch.cuda.synchronize()
            assert_close(from_layout(C, lc, lc), want, name=f'{la},{lb}->{lc} K={E}')


@pytest.mark.parametrize('B,L,H,E,expect_pair', [(8, 512, 16, 1024, True), (2, 128, 4, 256, False)])
def test_two_contractions_in_one_call(B, L, H, E, expect_pair):
    """sub_op_einsum_pair: a data gradient (with and without a residual added in its
    epilogue) and the weight gradient next to it, as one launch at the bench workload's
    sizes, and at small sizes (paired or not, as the launcher decides); either way against
    numpy.einsum and equal to what the two single calls give (to rounding where a
    small output's contraction is split differently)."""
    from substation_amd.ops import Ops
    o = Ops(B, L, H, E)
    sz = o.sizes
    rng = np.random.default_rng(11)
    mk = lambda lay, s=1.0: h16(s * rng.normal(size=tuple(sz[d] for d in lay)))
    nan = lambda lay: torch.full(tuple(sz[d] for d in lay), float('nan'), dtype=torch.float16, device='cuda')
    cases = [
        # dXlin1 + dWlin1
        (('BJU', 'UI', 'BJI', None), ('BJU', 'BJI', 'UI')),
        # dXQKV + residual, dWQKV
        (('QHPI', 'QBJHP', 'BJI', 'BJI'), ('QBJHP', 'BJI', 'QHPI')),
        # dXout, dWout
        (('IHP', 'BJI', 'BJHP', None), ('BJI', 'BJHP', 'IHP')),
    ]
    for (la1, lb1, lc1, lt1), (la2, lb2, lc2) in cases:
        # the shared operand is the same tensor in both products, as in a backward pass
        shared = {}
        def operand(lay, s=1.0):
            if lay not in shared:
                shared[lay] = mk(lay, s)
            return shared[lay]
        A1, B1 = operand(la1, 0.5), operand(lb1, 0.5)
        A2, B2 = operand(la2, 0.5), operand(lb2, 0.5)
        T1 = mk(lt1) if lt1 else None
        want1 = np.einsum(f'{la1},{lb1}->{lc1}'.lower(), A1, B1) + (T1 if lt1 else 0)
        want2 = np.einsum(f'{la2},{lb2}->{lc2}'.lower(), A2, B2)
        dev = {k: to_layout(v, k, k) for k, v in shared.items()}
        t1 = to_layout(T1, lt1, lt1) if lt1 else None
        C1, C2 = nan(lc1), nan(lc2)
        first = (dev[la1], la1, dev[lb1], lb1, C1, lc1) + ((t1, lt1) if lt1 else ())
        paired = o.einsum_pair(first, (dev[la2], la2, dev[lb2], lb2, C2, lc2))
        torch.cuda.synchronize()
        S1, S2 = nan(lc1), nan(lc2)
        o.einsum(dev[la1], la1, dev[lb1], lb1, S1, lc1, addend=t1, l_addend=lt1)
        o.einsum(dev[la2], la2, dev[lb2], lb2, S2, lc2)
        torch.cuda.synchronize()
        name = f'{la1},{lb1}->{lc1} + {la2},{lb2}->{lc2}'
        assert_close(from_layout(C1, lc1, lc1), want1, name=name + ' (first)')
        assert_close(from_layout(C2, lc2, lc2), want2, name=name + ' (second)')
        assert_close(C1.float().cpu().numpy(), S1.float().cpu().numpy(), tol=2e-3, name=name + ' first vs single')
        assert_close(C2.float().cpu().numpy(), S2.float().cpu().numpy(), tol=2e-3, name=name + ' second vs single')
    if expect_pair:
        # the pair the layer itself launches must have gone out as one launch here too
        la1, lb1, lc1 = 'BJU', 'UI', 'BJI'
        la2, lb2, lc2 = 'BJU', 'BJI', 'UI'
        d = {k: to_layout(mk(k, 0.5), k, k) for k in ('BJU', 'UI', 'BJI')}
        assert o.einsum_pair((d['BJU'], 'BJU', d['UI'], 'UI', nan('BJI'), 'BJI'),
                             (d['BJU'], 'BJU', d['BJI'], 'BJI', nan('UI'), 'UI'))


@pytest.mark.parametrize('L,E,U', [(8, 8, 8), (72, 136, 200), (64, 64, 3072), (1000, 72, 776), (2616, 128, 776), (1928, 72, 2056)])
def test_tiles_with_remainders(L, E, U):
    """Every operand orientation on tiles of each size (64 x 64 for few outputs up to 256 x 128 for many), with
    remainders in m, n and k; a bias row and a whole addend."""
    from substation_amd.ops import Ops
    o = Ops(1, L, 1, E, intermediate_size=U)
    sz = o.sizes
    rng = np.random.default_rng(L)
    mk = lambda lay: h16(rng.normal(size=tuple(sz[d] for d in lay)))
    for las, lbs, lc, bias in ((('BJI', 'IBJ'), ('UI', 'IU'), 'BJU', 'U'), (('BJU', 'UBJ'), ('UI', 'IU'), 'BJI', 'BJI')):
        for la in las:
            for lb in lbs:
                A, Bm, T = mk(la), mk(lb), mk(bias)
                want = np.einsum(f'{la},{lb}->{lc}'.lower(), A, Bm)
                C = torch.full(tuple(sz[d] for d in lc), float('nan'), dtype=torch.float16, device='cuda')
                assert o.handle.classify(la, lb, lc)['kernel'] == 1
                o.einsum(to_layout(A, la, la), la, to_layout(Bm, lb, lb), lb, C, lc)
                torch.cuda.synchronize()
                assert_close(from_layout(C, lc, lc), want, name=f'{la},{lb}->{lc}')
                o.einsum(to_layout(A, la, la), la, to_layout(Bm, lb, lb), lb, C, lc, addend=to_layout(T, bias, bias), l_addend=bias)
                torch.cuda.synchronize()
                assert_close(from_layout(C, lc, lc), want + T, name=f'{la},{lb}->{lc} + {bias}')


@pytest.mark.parametrize('B,L,H,E,U', [(1, 72, 3, 192, 776), (2, 1000, 2, 128, 512), (1, 2616, 12, 768, 776), (1, 2616, 12, 768, 3072)])
def test_products_sharing_a_launch(B, L, H, E, U):
    """A data gradient with a residual and a weight gradient as one list of tiles: remainders, several
    batches, contractions of unequal length, and more tiles than the chip takes at once."""
    from substation_amd.ops import Ops
    o = Ops(B, L, H, E, intermediate_size=U)
    sz = o.sizes
    g = torch.Generator(device='cuda').manual_seed(L)
    mk = lambda lay: torch.randn(tuple(sz[d] for d in lay), generator=g, device='cuda').half() * 0.5
    nan = lambda lay: torch.full(tuple(sz[d] for d in lay), float('nan'), dtype=torch.float16, device='cuda')
    for (la1, lb1, lc1, lt1), (la2, lb2, lc2) in (
            (('BJU', 'UI', 'BJI', 'BJI'), ('BJU', 'BJI', 'UI')),
            (('QHPI', 'QBJHP', 'BJI', 'BJI'), ('QBJHP', 'BJI', 'QHPI'))):
        d = {lay: mk(lay) for lay in {la1, lb1, la2, lb2}}
        T, C1, C2 = mk(lt1), nan(lc1), nan(lc2)
        o.einsum_pair((d[la1], la1, d[lb1], lb1, C1, lc1, T, lt1), (d[la2], la2, d[lb2], lb2, C2, lc2))
        torch.cuda.synchronize()
        w1 = np.einsum(f'{la1},{lb1}->{lc1}'.lower(), d[la1].double().cpu(), d[lb1].double().cpu(), optimize=True) + T.double().cpu().numpy()
        w2 = np.einsum(f'{la2},{lb2}->{lc2}'.lower(), d[la2].double().cpu(), d[lb2].double().cpu(), optimize=True)
        assert_close(C1.double().cpu().numpy(), w1, name=f'{la1},{lb1}->{lc1}')
        assert_close(C2.double().cpu().numpy(), w2, name=f'{la2},{lb2}->{lc2}')


@pytest.mark.parametrize('B,L,E,U', [(1, 4104, 1024, 4104), (4, 1000, 1032, 4096), (13, 208, 2048, 8192)])
def test_wide_tiles_with_remainders(B, L, E, U):
    """256 x 256 tiles whose last row and column of tiles are not whole, a contraction that is not a multiple of 64 where
    neither operand lies along it, an outer and an inner contraction, several tiles per workgroup, a scale, a bias row and
    a whole addend, and a data gradient beside a weight gradient (the two ways of reading A in one launch).  fp16
    operands, fp32 sums, one rounding: 2^-11 of the value, and sums of up to 8192 terms to 1e-5 of their rms."""
    from substation_amd.ops import Ops
    o = Ops(B, L, 8, E, intermediate_size=U)
    sz = o.sizes
    g = torch.Generator(device='cuda').manual_seed(E)
    mk = lambda lay: torch.randn(tuple(sz[d] for d in lay), generator=g, device='cuda').half()
    nan = lambda lay: torch.full(tuple(sz[d] for d in lay), float('nan'), dtype=torch.float16, device='cuda')

    def want(la, A, lb, Bm, lc, alpha=1.0, T=None, lt=None):
        k = [d for d in la if d in lb and d not in lc]
        ma, nb = [d for d in la if d in lc], [d for d in lb if d in lc]
        mat = lambda X, l, r, c: X.double().permute([l.index(d) for d in r + c]).reshape(int(np.prod([sz[d] for d in r])), -1)
        W = (alpha * torch.mm(mat(A, la, ma, k), mat(Bm, lb, k, nb))).half()
        W = W.reshape([sz[d] for d in ma + nb]).permute([(ma + nb).index(d) for d in lc])
        if T is None:
            return W.double()
        return W.double() + T.double().reshape([sz[d] if d in lt else 1 for d in lc])

    def check(C, W, name):
        err = (C.double() - W).abs() - 2.0 ** -10 * W.abs()
        assert float(err.max()) <= 2e-3 * float(W.pow(2).mean().sqrt()), name

    ways = [('BJI', 'UI'), ('BJI', 'IU'), ('IBJ', 'IU'), ('IBJ', 'UI')]
    for la, lb in ways if E % 64 == 0 else ways[2:3]:
        A, Bm, bias, T = mk(la), mk(lb), mk('U'), mk('BJU')
        for alpha, t, lt in ((1.0, None, None), (0.125, None, None), (1.0, bias, 'U'), (1.0, T, 'BJU')):
            C = nan('BJU')
            o.einsum(A, la, Bm, lb, C, 'BJU', alpha=alpha, addend=t, l_addend=lt)
            torch.cuda.synchronize()
            check(C, want(la, A, lb, Bm, 'BJU', alpha, t, lt), f'{la},{lb}->BJU alpha {alpha} + {lt}')
    if E == 2048:
        for (la1, lb1, lc1, lt1), (la2, lb2, lc2) in (
                (('BJU', 'UI', 'BJI', 'BJI'), ('BJU', 'BJI', 'UI')),
                (('QHPI', 'QBJHP', 'BJI', 'BJI'), ('QBJHP', 'BJI', 'QHPI'))):
            d = {lay: mk(lay) for lay in {la1, lb1, la2, lb2}}
            T, C1, C2 = mk(lt1), nan(lc1), nan(lc2)
            o.einsum_pair((d[la1], la1, d[lb1], lb1, C1, lc1, T, lt1), (d[la2], la2, d[lb2], lb2, C2, lc2))
            torch.cuda.synchronize()
            check(C1, want(la1, d[la1], lb1, d[lb1], lc1, 1.0, T, lt1), f'{la1},{lb1}->{lc1}')
            check(C2, want(la2, d[la2], lb2, d[lb2], lc2), f'{la2},{lb2}->{lc2}')


class _Guarded:
    """Tensors in the middle of allocations of their own: 4 MiB of a pattern on both sides, more than a tile of 256 rows of the
    outputs below, which no kernel may write and whose values (NaN as halves) no output may show."""
    GUARD = 4 << 20

    def __init__(self):
        self.held = []

    def place(self, shape, dtype=torch.float16, values=None):
        n = int(np.prod(shape)) * torch.empty(0, dtype=dtype).element_size()
        flat = torch.full((n + 2 * self.GUARD,), 0x7E, dtype=torch.uint8, device='cuda')
        self.held.append(flat)
        t = flat[self.GUARD:self.GUARD + n].view(dtype).view(shape)
        return t if values is None else t.copy_(values)

    def check(self, name):
        torch.cuda.synchronize()
        for i, flat in enumerate(self.held):
            assert bool((flat[:self.GUARD] == 0x7E).all()) and bool((flat[-self.GUARD:] == 0x7E).all()), (name, i)


@pytest.mark.parametrize('L,E,U', [(4104, 1024, 4104),     # 256 x 256 tiles whose last row and column have 8 of 256
                                   (4296, 1032, 4240),     # 200 rows, 144 columns; a contraction with a remainder
                                   (2616, 128, 776), (1928, 72, 2056), (72, 136, 200)])
def test_nothing_behind_an_output_is_written_and_nothing_behind_an_operand_read(L, E, U):
    """Rows and columns of tiles that the output has not: every way of reading the operands, alone, with a bias row and with
    a whole addend."""
    from substation_amd.ops import Ops
    o = Ops(1, L, 1, E, intermediate_size=U)
    sz = o.sizes
    g = torch.Generator(device='cuda').manual_seed(L)
    for la in ('BJI', 'IBJ'):
        for lb in ('UI', 'IU'):
            mem = _Guarded()
            mk = lambda lay: mem.place([sz[d] for d in lay], values=torch.randn([sz[d] for d in lay], generator=g, device='cuda'))
            A, Bm, bias, T = mk(la), mk(lb), mk('U'), mk('BJU')
            mat = lambda X, lay: X.float().reshape(L, E) if lay == 'BJI' else X.float().reshape(E, -1).t() if lay == 'IBJ' else \
                X.float() if lay == 'IU' else X.float().t()
            want = mat(A, la) @ mat(Bm, lb)
            for t, lt in ((None, None), (bias, 'U'), (T, 'BJU')):
                C = mem.place([sz[d] for d in 'BJU'])
                o.einsum(A, la, Bm, lb, C, 'BJU', addend=t, l_addend=lt)
                name = f'{la},{lb} + {lt}'
                mem.check(name)
                w = want if t is None else want + t.float().reshape(-1, U)
                # fp16 outputs of sums of up to 1032 terms: half a step, twice with an addend, and the sums' order
                assert float((C.float().reshape(L, U) - w).abs().max()) <= 2.0 ** -10 * float(w.abs().max()), name


@pytest.mark.parametrize('L,E,U', [(4104, 1024, 4128), (2616, 768, 3104), (1000, 512, 4128)])
@pytest.mark.parametrize('act', ['relu', 'gelu'])
def test_nothing_behind_what_an_activation_epilogue_leaves_is_written(L, E, U, act):
    """The output, the pre-activation, the bits and the gradient of tiles that are not whole."""
    from substation_amd.ops import Ops
    o = Ops(1, L, E // 64, E, intermediate_size=U, activation=act, seed=7)
    sz = o.sizes
    g = torch.Generator(device='cuda').manual_seed(L)
    mem = _Guarded()
    mk = lambda lay, s=1.0: mem.place([sz[d] for d in lay], values=s * torch.randn([sz[d] for d in lay], generator=g, device='cuda'))
    x, w1, bias, dy, w2 = mk('BJI'), mk('UI', 0.05), mk('U'), mk('BJI'), mk('IU', 0.05)
    out, lin, dlin = (mem.place([sz[d] for d in 'BJU']) for _ in range(3))
    bits, dbias = mem.place([L * U // 8], torch.uint8), mem.place([U])
    assert o.einsum_bad(x, 'BJI', w1, 'UI', bias, 'U', lin if act == 'gelu' else None, out, 'BJU', bits, p=0.1)
    mem.check('forward')
    assert o.einsum_bdrlb(dy, 'BJI', w2, 'IU', lin if act == 'gelu' else out, 'BJU', bits, dlin, 'BJU', dbias)
    mem.check('backward')
    # and the values are those of the operators, the bias gradient to rounding (up to 4104 terms in another order)
    sb, mask, lin2, out2, dlin2, dbias2 = (torch.empty(shape, dtype=torch.float16, device='cuda') for shape in [out.shape] * 5 + [[U]])
    o.einsum(x, 'BJI', w1, 'UI', sb, 'BJU')
    o.bad(sb, 'BJU', bias, lin2, 'BJU', mask, 'BJU', out2, 'BJU', p=0.1)
    o.einsum(dy, 'BJI', w2, 'IU', sb, 'BJU')
    o.bdrlb(sb, 'BJU', mask, 'BJU', lin2, 'BJU', dlin2, 'BJU', dbias2)
    assert torch.equal(out, out2) and torch.equal(dlin, dlin2) and float(dlin.float().abs().max()) > 0
    assert_close(dbias.float().cpu().numpy(), dbias2.float().cpu().numpy(), tol=2e-3, name='dbias')


# (orders: words along k, along the rows and neither, of either operand; an output that is contiguous along m; steps of 32 k with one, 31 and no
# k left over, tiles of 128 x 64 with 1, 32, 33 and 64 columns in the last one)
@pytest.mark.parametrize('la,lb,lc', [('BJHP', 'BKHP', 'HBJK'), ('HBJK', 'BKHP', 'BJHP'), ('HBKJ', 'KBHP', 'BJHP'), ('HPBJ', 'BKHP', 'BHKJ'),
                                      ('BHJP', 'HBPK', 'JBHK'), ('BHJK', 'BJHP', 'HBPK')])
# (up to 24 k in steps of 8: 1 to 24 positions; products of up to 64 rows in tiles of 64: 1, 32, 33, 64)
@pytest.mark.parametrize('dims', [(2, 33, 2, 24), (1, 97, 1, 64), (1, 129, 3, 192), (3, 65, 1, 31), (1, 255, 1, 8), (2, 1, 2, 10), (1, 8, 2, 66),
                                  (2, 9, 1, 64), (3, 24, 2, 50), (1, 25, 2, 48), (2, 32, 1, 17), (1, 64, 2, 130), (2, 63, 3, 3)])
def test_sums_without_whole_words_are_one_chain_of_fused_multiply_adds(la, lb, lc, dims):
    """Bit for bit, in the order of k: products of halves are exact in float64, and so are their sums with an fp32 value (here: 11 + 11
    bits at exponents within 2 ** +-24), so that rounding each sum to float32 is what fmaf does."""
    from substation_amd.ops import Ops
    o = Ops(*dims)
    sz = o.sizes
    if o.handle.classify(la, lb, lc)['kernel'] == 1:
        pytest.skip('whole words')
    rng = np.random.default_rng(len(la) + dims[1])
    draw = lambda l: h16(np.clip(rng.normal(size=tuple(sz[d] for d in l)), -4, 4)) * (rng.random(size=tuple(sz[d] for d in l)) > 0.1)
    A, B = draw(la).astype(np.float64), draw(lb).astype(np.float64)
    k, = set(la) & set(lb) - set(lc)
    acc = np.zeros(tuple(sz[d] for d in lc), np.float32)
    for i in range(sz[k]):
        a, b = np.take(A, i, la.index(k)), np.take(B, i, lb.index(k))
        term = np.einsum(f'{la.replace(k, "")},{lb.replace(k, "")}->{lc}'.lower(), a, b)
        acc = (acc.astype(np.float64) + term).astype(np.float32)
    C = torch.full(tuple(sz[d] for d in lc), float('nan'), dtype=torch.float16, device='cuda')
    half = lambda x: torch.from_numpy(x.astype(np.float16)).cuda()
    o.einsum(half(A), la, half(B), lb, C, lc)
    torch.cuda.synchronize()
    assert (C.cpu().numpy().view(np.uint16) == acc.astype(np.float16).view(np.uint16)).all()
