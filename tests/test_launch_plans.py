"""Which launches a call makes, and that what is kept from one call to the next does not change them (on the CPU: tests/launches.py)."""
import copy
import ctypes
import itertools
import re

import pytest

import tests.launches as launches


def _pointers(addresses):
    return (ctypes.c_void_p * len(addresses))(*addresses), len(addresses)


def _pass(lib, check, handle):
    """The launches of a forward and a backward call (layer calls with 37 and 64 tensors, all of them aligned)."""
    forward = launches.tensors(37)
    backward = launches.tensors(64, first=64)
    return launches.launched(lambda: (check(lib.sub_encoder_forward(handle.ptr, *_pointers(forward))),
                                      check(lib.sub_encoder_backward(handle.ptr, *_pointers(backward)))))


def _orders(L, which):
    lay = copy.deepcopy(L.mi355x_layouts() if which == 'own' or which == 'token-contiguous'
                        else L.reference_layouts('bert-b8-l512-h16-e1024'))
    # feed-forward tensors with the tokens contiguous: weight gradients whose operands both lie along their contraction
    other = {'token-contiguous': dict(DLIN1='UBJ', DROP2='UBJ', LIN1='UBJ', SB1='IBJ', DLIN2='IBJ', WKQV='QIHP'),
             'reference-but-LINW1': dict(LINW1='UI')}.get(which, {})
    for group in ('params', 'forward_interm', 'backward_interm'):
        lay[group] = [(name, other.get(name, order)) for name, order in lay[group]]
    return lay


def _options_between_passes():
    from substation_amd import _lib, layouts as L
    lib = _lib.load()
    # (weight gradients over 4096 tokens, over 4000, which is no multiple of 64, and over 215, which is none of 8)
    for which, (B, S, H, E) in itertools.product(('own', 'reference', 'reference-but-LINW1', 'token-contiguous'),
                                                 ((8, 512, 16, 1024), (8, 500, 16, 1024), (5, 43, 4, 256))):
        for option, value in ((11, 0), (11, 1), (5, 0), (7, 0), (3, 0), (1, 0), (2, 0), (4, 0), (12, 1)):
            def handle():
                return _lib.Handle(_lib.make_config(B, S, H, E, _orders(L, which), 0.1, 0.1, 0.1, 0.1, activation='gelu'))
            fresh, used = handle(), handle()
            if (option, value) == (11, 1):
                used.set_option(11, 0)
            _pass(lib, _lib.check, used)
            used.set_option(option, value)
            fresh.set_option(option, value)
            try:
                got, want = _pass(lib, _lib.check, used), _pass(lib, _lib.check, fresh)
                at = next((i for i, (a, b) in enumerate(itertools.zip_longest(got, want)) if a != b), None)
                print('same' if at is None else f'{which} {B}x{S} option {option}={value}: {got[at:at + 1]} for {want[at:at + 1]}')
            except _lib.SubstationError as e:
                print(f'{which} {B}x{S} option {option}={value}: {e}')


def test_options_that_change_between_passes(tmp_path):
    """A handle whose options change after a pass launches what one does that had them from the start."""
    lines = launches.run(_options_between_passes, tmp_path)
    assert len(lines) == 4 * 3 * 9 and set(lines) == {'same'}, [l for l in lines if l != 'same']


# the ten products that a decoder layer has at the end of its backward pass: layouts of A, B, C and of an addend; which of its two
# sequence lengths they are over
GROUP = [('QHPI', 'QBJHP', 'BJI', 'BJI', 0), ('BKHP', 'HPI', 'BKI', 'BKI', 1), ('BKHP', 'BKI', 'HPI', None, 1),
         ('BKHP', 'BKI', 'HPI', None, 1), ('QBJHP', 'BJI', 'QHPI', None, 0), ('BJI', 'BJHP', 'IHP', None, 0),
         ('BJHP', 'BJI', 'HPI', None, 0), ('BJI', 'BJHP', 'IHP', None, 0), ('BJU', 'BJI', 'UI', None, 0), ('BJI', 'BJU', 'IU', None, 0)]


class Group:
    """GROUP as a call on a handle of one size, some of the products by another handle's."""

    def __init__(self, B=8, S=256, H=16, E=1024, source=512, options=()):
        from substation_amd import _lib, layouts as L
        self.l, self.lib = _lib, _lib.load()
        self.handles = [_lib.Handle(_lib.make_config(B, s, H, E, L.mi355x_layouts())) for s in (S, source)]
        for option, value in options:
            self.handles[0].set_option(option, value)
        self.products = (_lib.Einsum * len(GROUP))()
        at = itertools.count(1)
        for q, (la, lb, lc, lt, which) in zip(self.products, GROUP):
            q.sizes = self.handles[which].ptr
            q.A, q.B, q.C = (next(at) << 36 for _ in range(3))
            q.l_A, q.l_B, q.l_C = la.encode(), lb.encode(), lc.encode()
            if lt:
                q.T, q.l_T = q.C, lt.encode()
            q.alpha = 1.0

    def launched(self, on=None):
        """By its own handle or by the one of another group (the sizes stay its own)."""
        handle = (on or self).handles[0].ptr
        return launches.launched(lambda: self.l.check(self.lib.sub_op_einsum_group(handle, self.products, len(self.products))))


def _timed_operator_calls():
    from substation_amd import _lib
    g = Group()
    g.handles[0].profile_enable()
    for _ in range(5):
        g.launched()
        a, b = launches.tensors(2)
        _lib.check(g.lib.sub_op_relayout(g.handles[0].ptr, a, b'BJI', b, b'IBJ'))
    print(launches.recorder.recorder_events())


def test_operator_calls_leave_nothing_in_a_handles_timing(tmp_path):
    """Entries of the per-launch timing are begun anew by the next layer call; a handle that operator calls are made on has none."""
    assert launches.run(_timed_operator_calls, tmp_path) == ['0']


def _misaligned_members():
    for odd in (None, 2, 4, 9):          # (those without an addend: it is refused with one)
        g = Group()
        if odd is not None:
            g.products[odd].B += 2
        names = [name for name, _ in g.launched()]
        print(sum('k_gemm_fma' in n for n in names), sum('ILi7E' in n or 'Li7ELi' in n for n in names), len(names))


def test_a_misaligned_member_of_a_group_runs_alone(tmp_path):
    """One product that the tiles do not take (an operand that is an odd slice of a buffer): a launch more, and no others'."""
    lines = [tuple(int(x) for x in l.split()) for l in launches.run(_misaligned_members, tmp_path)]
    whole, *rest = lines
    assert whole[0] == 0 and whole[1] >= 1
    for scalar, shared, total in rest:
        assert scalar == 1 and shared >= 1 and total <= whole[2] + 1


def _groups_in_turn():
    def groups():
        for dims in ((8, 256, 16, 1024, 512), (2, 128, 12, 768, 128), (3, 40, 4, 256, 72), (16, 384, 12, 768, 256), (4, 1000, 16, 1024, 96)):
            for odd in (None, 4):
                g = Group(*dims)
                if odd is not None:
                    g.products[odd].B += 2
                yield g
    want = [g.launched() for g in groups()]
    one = Group()
    for on in (1, 0, 1):
        one.handles[0].set_option(5, on)
        for turn in range(2):
            for g, w in zip(groups(), want):
                got = g.launched(one)
                alone = all('Li7E' not in name for name, _ in got)
                print('same' if (got == w if on else alone) else (on, turn, got, w))


def test_groups_that_a_handle_has_seen_before(tmp_path):
    """More groups than a handle keeps plans of, by sizes, alignments and the option, over and over: what a new handle launches."""
    lines = launches.run(_groups_in_turn, tmp_path)
    assert len(lines) == 60 and set(lines) == {'same'}, [l for l in lines if l != 'same'][:2]


def _groups_in_a_block_of_sums():
    for streams in ((1, 1, 1), (1, 2, 1), (1, 2, 2), (1, 1, 2), (2, 2, 1)):        # of a sum, of the group, where the block ends
        g = Group()
        h = g.handles[0]
        a, b = launches.tensors(2, first=64)
        for turn in range(2):                # (the first one makes the buffer)
            h.set_stream(streams[0])
            h.defer_column_sums(True)
            g.l.check(g.lib.sub_op_baob(h.ptr, a, b'BJI', b))
            h.set_stream(streams[1])
            g.launched()

            def end():
                h.set_stream(streams[2])
                h.defer_column_sums(False)
            last = [name for name, _ in launches.launched(end)]
        print(streams, len(last))


def test_a_group_finishes_no_column_sums_of_another_stream(tmp_path):
    """It would not wait for them; they end with the block, on the stream that is current there."""
    lines = launches.run(_groups_in_a_block_of_sums, tmp_path)
    assert lines == ['(1, 1, 1) 0', '(1, 2, 1) 1', '(1, 2, 2) 1', '(1, 1, 2) 0', '(2, 2, 1) 0']


def _two_threads():
    import threading
    from substation_amd import _lib, layouts as L
    lib = _lib.load()
    h = _lib.Handle(_lib.make_config(2, 128, 4, 256, L.mi355x_layouts(), 0.1, 0.1, 0.1, 0.1, activation='gelu'))
    h.set_option(12, 1)
    forward, backward = _pointers(launches.tensors(37)), _pointers(launches.tensors(64, first=64))
    said, done = threading.Event(), threading.Event()
    refused = []

    def without_gradients():
        _lib.check(lib.sub_forward_alone(h.ptr))
        said.set()
        done.wait()
        _lib.check(lib.sub_encoder_forward(h.ptr, *forward))
        refused.append(lib.sub_encoder_backward(h.ptr, *backward) < 0)

    other = threading.Thread(target=without_gradients)
    other.start()
    said.wait()
    _lib.check(lib.sub_encoder_forward(h.ptr, *forward))
    print(lib.sub_encoder_backward(h.ptr, *backward) == 0)
    done.set()
    other.join()
    print(refused == [True])


def test_a_forward_pass_of_another_thread_keeps_what_its_backward_pass_reads(tmp_path):
    """That no backward call follows is said of the calling thread's next forward call, whatever another one calls in between."""
    assert launches.run(_two_threads, tmp_path) == ['True', 'True']


# (B, L, H, E): how the four forward products of a ReLU layer are summed (projections, out, lin1, lin2): in 256 x 256 tiles, whose k slices
# are twice as long (W), or in others (R), and in how many parts; and lin1 with its activation, which products in parts do not have
ORDERS = {
    (1, 16, 8, 512): 'R1 R1 R1 R4 R', (1, 64, 12, 768): 'R1 R1 R1 R6 R', (1, 64, 16, 1024): 'R2 R2 R2 R8 -',
    (2, 128, 12, 768): 'R1 R1 R1 R6 R', (4, 256, 12, 768): 'R1 R1 R1 R5 R', (24, 77, 12, 768): 'R1 R1 R1 R2 R',
    (13, 201, 12, 768): 'R1 R1 R1 R2 R', (8, 500, 16, 1024): 'W1 R1 W1 R1 W', (8, 512, 16, 1024): 'W1 R1 W1 R1 W',
    (10, 512, 16, 1024): 'W1 R1 R1 R1 R', (12, 512, 16, 1024): 'R1 R1 R1 R1 R', (16, 512, 16, 1024): 'R1 R1 W1 R1 W',
    (96, 128, 16, 1024): 'R1 W1 W1 W1 W', (1, 512, 16, 1024): 'R2 R2 R2 R8 -', (2, 512, 16, 1024): 'R1 R2 R1 R4 R',
    (1, 128, 32, 4096): 'R2 R8 R2 R8 -', (1, 512, 32, 4096): 'R1 R2 R1 R2 R', (2, 1024, 16, 2048): 'W1 R1 W1 R1 W',
    (4, 2048, 32, 4096): 'W1 W1 W1 W1 W', (7, 640, 16, 2048): 'W1 W1 R1 W1 R', (9, 333, 12, 768): 'R1 R1 W1 R1 W',
    (5, 1000, 16, 1024): 'W1 R1 R1 R1 R', (40, 200, 8, 512): 'W1 R1 W1 R1 W',
}


def _orders_in_front_of_a_relu():
    from substation_amd import _lib, layouts as L
    lib = _lib.load()
    for B, S, H, E in ORDERS:
        h = _lib.Handle(_lib.make_config(B, S, H, E, L.mi355x_layouts(), 0.1, 0.1, 0.1, 0.1, activation='relu'))
        h.set_option(12, 1)
        row = []
        for la, lb, lc in (('BJI', 'QHPI', 'QBJHP'), ('IHP', 'BJHP', 'BJI'), ('BJI', 'UI', 'BJU'), ('BJU', 'IU', 'BJI')):
            a, b, c = launches.tensors(3)
            (name, grid), *reduction = launches.launched(lambda: _lib.check(
                lib.sub_op_einsum(h.ptr, a, la.encode(), b, lb.encode(), c, lc.encode(), 1.0)))
            wide = 'k_gemm_wide' in name
            parts = 1
            if reduction:                                   # (a workgroup for each part of a tile)
                tm, tn, wm, wn = (int(x) for x in re.findall(r'Li(\d+)E', name)[:4])
                shape = h.classify(la, lb, lc)
                tiles = -(-shape['M'] // (32 * tm * wm)) * -(-shape['N'] // (32 * tn * wn)) * shape['batch']
                assert grid[0] % tiles == 0
                parts = grid[0] // tiles
            row.append('RW'[wide] + str(parts))
        forward = launches.launched(lambda: _lib.check(lib.sub_encoder_forward(h.ptr, *_pointers(launches.tensors(37)))))
        act = ['RW'['k_gemm_wide' in n] for n, _ in forward if re.search(r'k_gemm_(ring|wide).*Li[13]EEEv', n)]
        print(' '.join(row + (act or ['-'])))


def test_order_of_the_sums_in_front_of_a_relu(tmp_path):
    """It is a fixed function of the shape: another one moves gates, and with them whole rows of gradients."""
    lines = launches.run(_orders_in_front_of_a_relu, tmp_path)
    assert dict(zip(ORDERS, lines)) == ORDERS


HALVES_TESTED = [(128, 128), (256, 128), (128, 384), (512, 512), (384, 1024)]

# (samples, heads, queries, keys, head size, mask, activation): blocks of 128 queries and of keys; whether forward, dQ, and dK and dV take the
# kernels in which two waves share a block's other side (h) or those of whole blocks (w)
ATTENTION = {
    (2, 16, 512, 512, 64, False, 'gelu'): 'hhh',      # 128 blocks
    (3, 12, 512, 512, 64, False, 'gelu'): 'www',      # 144
    (8, 16, 128, 512, 64, False, 'gelu'): 'hhw',      # 128 of queries, 512 of keys
    (2, 16, 512, 512, 64, False, 'relu'): 'whh',
    (2, 16, 512, 512, 64, True, 'relu'): 'whh',
    (2, 16, 512, 512, 128, False, 'gelu'): 'www',
    (4, 12, 384, 384, 64, True, 'gelu'): 'hhh',       # 144 blocks of 12 tiles
    (4, 16, 512, 512, 64, True, 'gelu'): 'hhh',       # 256 of 16
    (2, 16, 1024, 1024, 64, True, 'gelu'): 'hhh',     # 256 of 32
    (8, 16, 256, 256, 64, True, 'gelu'): 'www',       # 256 of 8
    (9, 8, 512, 512, 64, True, 'gelu'): 'www',        # 288 of 16
    (3, 12, 1024, 1024, 64, True, 'gelu'): 'hhw',     # 288 of 32
    (2, 12, 2048, 2048, 64, True, 'gelu'): 'hhw',     # 384 of 64
    (25, 16, 128, 1024, 64, True, 'gelu'): 'www',     # 400 of queries, 3200 of keys
    (2, 24, 128, 384, 64, True, 'gelu'): 'hhw',       # 48 of queries; 144 of keys, of 4 tiles
    (2, 16, 1000, 1000, 64, True, 'gelu'): 'hhh',     # (a layer's: lengths with an end inside a tile)
    (5, 10, 201, 201, 64, False, 'gelu'): 'hhh',      # 100
    (13, 12, 201, 201, 64, False, 'gelu'): 'www',     # 312
    # what tests/test_ops_gpu.py takes for halves and for whole blocks
    **{(2, 2, J, K, 64, mask, 'gelu'): 'hhh' for J, K in HALVES_TESTED for mask in (False, True)},
    **{(130, 2, J, K, 64, mask, 'gelu'): 'www' for J, K in HALVES_TESTED for mask in (False, True)},
    **{(n, 2, L, L, 64, True, 'gelu'): row for L, few in ((97, 2), (400, 20), (1001, 12)) for n, row in ((few, 'hhh'), (70, 'www'))},
}


def _attention_launches():
    from substation_amd import _lib, layouts as L
    lib = _lib.load()
    for (B, H, J, K, P, mask, act) in ATTENTION:
        h = _lib.Handle(_lib.make_config(B, J, H, H * P, L.mi355x_layouts(), 0.1, 0.1, 0.1, 0.1, activation=act))
        q, k, v, out, dout, dq, dk, dv, m, bq, bk, bv, stats, keep = launches.tensors(14)
        m = m if mask else None
        calls = []
        if J % 128 == 0 and K % 128 == 0:
            calls.append(lambda: (
                _lib.check(lib.sub_op_attention_forward(h.ptr, J, K, q, b'BJHP', k, v, b'BKHP', out, b'BJHP', stats, keep, m, b'JK', 0.125, 0.1, 0)),
                _lib.check(lib.sub_op_attention_backward_biases(h.ptr, J, K, q, b'BJHP', k, v, b'BKHP', out, b'BJHP', dout, b'BJHP', stats, keep, dq,
                                                                b'BJHP', dk, dv, b'BKHP', m, b'JK', 0.125, bq, bk, bv))))
        if J == K:
            if mask:
                h.set_attention_mask(m, 'JK')
            calls.append(lambda: (_lib.check(lib.sub_encoder_forward(h.ptr, *_pointers(launches.tensors(37)))),
                                  _lib.check(lib.sub_encoder_backward(h.ptr, *_pointers(launches.tensors(64, first=64))))))
        blocks = lambda n: B * H * -(-n // 128)
        seen = set()
        for call in calls:
            row = ''
            for name, (grid, *_) in launches.launched(call):
                kernel = re.search(r'k_mha_(fwd|bwd_dq|bwd_dkv)(_halves)?ILi(\d+)ELb(\d)ELb(\d)E', name)
                if not kernel:
                    continue
                which, halves, p, masked, any_length = kernel.groups()
                whole = blocks(K if which == 'bwd_dkv' else J)
                assert (int(p), int(masked)) == (P, mask) and grid == whole * (2 if halves else 1)
                # (two workgroups on a CU: not the one whose waves have a SIMD to themselves; see tests/test_kernel_registers.py)
                ends = J % 128 != 0 or K % 128 != 0
                assert int(any_length) == (ends or bool(halves and which == 'bwd_dkv' and mask and whole > 128))
                row += 'h' if halves else 'w'
            seen.add(row)
        print(' '.join(sorted(seen)))


def test_which_attention_launches_share_a_block_between_two_waves(tmp_path):
    """Operators and layers alike: up to 128 blocks, behind a mask up to one for each of 256 CUs where a block has 12 tiles to walk, but
    for dK and dV up to one and a half where it has 32."""
    lines = launches.run(_attention_launches, tmp_path)
    assert dict(zip(ATTENTION, lines)) == ATTENTION


# rows, features: rows to a workgroup of k_bdrln_flat (one row: either)
BDRLN = {(4, 768): 4, (16, 768): 4, (17, 768): 1, (255, 768): 1, (256, 768): 4, (16, 2048): 4, (16, 2056): 1, (8, 4096): 1}
# rows, features: waves and workgroups of k_lnbwd_flat, for two sums and for four
LNBWD = {(1, 512): '4:1 4:1', (512, 512): '4:128 4:128', (513, 512): '8:65 8:65', (1536, 512): '8:192 8:192', (1537, 512): '16:97 8:193',
         (1024, 520): '4:256 4:256', (1025, 520): '8:129 8:129', (2048, 1024): '8:256 8:256', (2049, 1024): '16:129 8:256', (8192, 1024): '16:256 8:256'}
# positions, head size: rows and k of the tiles of the scores' product, workgroups of four products
ANY_STRIDES = {(1, 10): '64 8 4', (63, 24): '64 8 4', (64, 25): '64 32 4', (65, 24): '128 8 8', (65, 25): '128 32 8', (201, 64): '128 32 32'}


def _few_rows_and_odd_products():
    from substation_amd import _lib, layouts as L
    lib = _lib.load()
    t = launches.tensors(16)

    def handle(*dims):
        return _lib.Handle(_lib.make_config(*dims, L.mi355x_layouts(), 0.1, 0.1, 0.1, 0.1))

    def only(kernel, call):
        (found, grid), = [(re.search(kernel, name), grid[0]) for name, grid in launches.launched(lambda: _lib.check(call())) if re.search(kernel, name)]
        return [int(n) for n in found.groups()] + [grid]

    for rows, features in BDRLN:
        h = handle(rows, 1, 1, features)
        grid, = only('k_bdrln_flat', lambda: lib.sub_op_bdrln(
            h.ptr, t[0], b'BJI', t[1], b'BJI', t[2], t[3], t[4], t[5], b'BJI', t[6], b'BJI', t[7], b'BJI', t[8], b'BJI', t[9], b'BJI', t[10], b'BJ', 0.1, 1))
        print({rows: 1, -(-rows // 4): 4}.get(grid))
    for rows, features in LNBWD:
        h, row = handle(rows, 1, 1, features), []
        for four in (False, True):
            second = [x if four else None for x in t[11:15]]
            waves, grid = only(r'k_lnbwd_flatILi\dELb\dELb\dELb\dELi1ELi(\d+)E', lambda: lib.sub_op_ln_backward(
                h.ptr, int(four), t[0], b'BJI', t[1], t[2], b'BJI', second[0], b'BJI', second[1], b'BJI', t[3], b'BJ', t[4], b'BJI', t[5], b'BJI', t[6],
                b'BJI', t[7], b'BJI', t[8], b'BJI', t[9], t[10], second[2], second[3]))
            row.append(f'{waves}:{grid}')
        print(*row)
    for n, size in ANY_STRIDES:
        h = handle(2, n, 2, 2 * size)
        print(*only(r'k_gemm_fmaILi\dELi\dELi(\d+)ELi(\d+)E',
                    lambda: lib.sub_op_einsum(h.ptr, t[0], b'BJHP', t[1], b'BKHP', t[2], b'HBJK', 1.0)))


def test_launches_of_few_rows_and_of_products_without_whole_words(tmp_path):
    """Where a rule changes its answer: nothing that a result shows (each was timed on both sides)."""
    lines = launches.run(_few_rows_and_odd_products, tmp_path)
    want = [str(v) for v in [*BDRLN.values(), *LNBWD.values(), *ANY_STRIDES.values()]]
    assert lines == want
