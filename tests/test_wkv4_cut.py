"""How the RWKV-4 scan is cut over the compute units: frhip_wkv4_cut, a function of the sizes alone."""
import ctypes as C
import importlib

import pytest

fr = importlib.import_module("faster-rwkv_amd")


def cut(T, channels, units=256):
    """-> channels of a workgroup, workgroups, blocks, chunks of a block, steps of a chunk"""
    out = (C.c_int * 5)()
    assert fr.lib().frhip_wkv4_cut(T, channels, units, out) == 0
    return tuple(out)


def test_every_width_fills_the_compute_units():
    """A workgroup is one compute unit's: from 2048 channels on nine of ten have one, whatever the width's divisors
    (4736 channels in 32s would be 148 workgroups), or as many rounds of them as 32 channels at most ask for."""
    for c in range(2048, 16385, 64):
        cg, groups, *_ = cut(1024, c)
        rounds = -(-c // 8192)
        assert 8 <= cg <= 32 and (groups - 1) * cg < c <= groups * cg
        assert 0.9 * 256 * rounds <= groups <= 256 * rounds, (c, cg, groups)


@pytest.mark.parametrize("c", [64, 768, 2048, 2112, 2560, 3584, 4096, 4736, 5120, 8192, 8256])
def test_time_is_covered_by_what_a_workgroup_holds(c):
    for t in list(range(1, 70)) + [127, 128, 129, 511, 1000, 1024, 1025, 1100, 2047, 2048, 2049, 4096, 4099, 8192, 30000]:
        cg, _, blocks, chunks, steps = cut(t, c)
        assert cg * chunks <= 1024 and 1 <= steps <= 16
        assert blocks * chunks * steps >= t
        assert (blocks - 1) * chunks * steps < t  # the last block is not empty


def test_arguments():
    out = (C.c_int * 5)()
    f = fr.lib().frhip_wkv4_cut
    assert f(4, 64, 256, None) == -1 and f(0, 64, 256, out) == f(4, 65, 256, out) == f(4, 64, 0, out) == -2
