"""Waves per SIMD that the attention kernels are built for, from the register counts in the library's own metadata: two or
three registers more halve them, and no other test would notice."""
import os
import re
import struct

import msgpack
import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'substation_amd', 'lib', 'libsubstation_amd.so')


def _kernels():
    """{mangled name: its metadata} of every code object in the library (AMDGPU ELF notes, MessagePack)."""
    if not os.path.exists(LIB):
        import __graft_entry__
        __graft_entry__.build()
    data, found, at = open(LIB, 'rb').read(), {}, 0
    while (at := data.find(b'\x7fELF', at + 1)) > 0:
        if struct.unpack_from('<H', data, at + 18)[0] != 224:        # EM_AMDGPU
            continue
        sections, = struct.unpack_from('<Q', data, at + 40)
        size, count = struct.unpack_from('<HH', data, at + 58)
        for i in range(count):
            kind, _, _, offset, length = struct.unpack_from('<IQQQQ', data, at + sections + i * size + 4)
            if kind != 7:                                            # SHT_NOTE
                continue
            name_len, desc_len, _ = struct.unpack_from('<III', data, at + offset)
            desc = at + offset + 12 + (name_len + 3) // 4 * 4
            for k in msgpack.unpackb(data[desc:desc + desc_len])['amdhsa.kernels']:
                found[k['.name']] = k
    return found


@pytest.fixture(scope='module')
def kernels():
    return _kernels()


#: (head size, masked, lengths that are no multiples of 128): waves of the forward, dQ, dK and dV kernels
WAVES = {(64, 0, 0): (3, 3, 2), (64, 0, 1): (3, 3, 2), (64, 1, 0): (2, 2, 2), (64, 1, 1): (3, 2, 2),
         (128, 0, 0): (2, 2, 1), (128, 0, 1): (2, 2, 1), (128, 1, 0): (1, 1, 1), (128, 1, 1): (1, 1, 1)}
#: those in which two waves share a block's other side: up to 256 workgroups without a mask, one on a CU; twice as many with one, two on a CU
#: (dK and dV then by the kernel for any length)
HALVES = {(0, 0): (2, 2, 2), (0, 1): (2, 2, 2), (1, 0): (2, 2, 1), (1, 1): (2, 2, 2)}


@pytest.mark.parametrize('variant', sorted(WAVES))
def test_waves_per_simd_of_the_attention_kernels(kernels, variant):
    for kernel, waves in zip(('k_mha_fwd', 'k_mha_bwd_dq', 'k_mha_bwd_dkv'), WAVES[variant]):
        p, masked, ragged = variant
        which = [k for n, k in kernels.items() if re.search(rf'{kernel}ILi{p}ELb{masked}ELb{ragged}E', n)]
        assert len(which) == 1
        k = which[0]
        # 512 registers per SIMD and lane, in blocks of 8; vgpr_count is vector and accumulation registers together
        assert 512 // ((k['.vgpr_count'] + 7) // 8 * 8) >= waves, (kernel, variant, k['.vgpr_count'])


@pytest.mark.parametrize('variant', sorted(HALVES))
def test_waves_per_simd_of_the_attention_kernels_by_halves(kernels, variant):
    for kernel, waves in zip(('k_mha_fwd_halves', 'k_mha_bwd_dq_halves', 'k_mha_bwd_dkv_halves'), HALVES[variant]):
        masked, ragged = variant
        which = [k for n, k in kernels.items() if re.search(rf'{kernel}ILi64ELb{masked}ELb{ragged}E', n)]
        assert len(which) == 1
        k = which[0]
        assert 512 // ((k['.vgpr_count'] + 7) // 8 * 8) >= waves, (kernel, variant, k['.vgpr_count'])
        assert k['.vgpr_spill_count'] == 0, (kernel, variant)
