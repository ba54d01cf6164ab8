"""Node tiles per wave of the general convolution, chosen on the host: the
measured side of every line of slbn_conv_ntw and slbn_conv_ci."""
import ctypes as C
import os

import pytest

from conftest import ROOT

LIB = os.path.join(ROOT, "sunlightlb_amd", "libsunlightlb.so")


@pytest.mark.parametrize("cin,cout,nodes,tiles,ci", [
    (64, 64, 1080, 1, 64), (64, 64, 14400, 1, 64), (64, 64, 30000, 2, 64), (64, 64, 39600, 4, 64),
    (64, 64, 50400, 4, 64), (64, 64, 125000, 4, 64), (64, 16, 50400, 4, 64), (16, 32, 125000, 4, 16),
    (16, 16, 69120, 2, 16), (32, 16, 69120, 2, 32), (16, 16, 125000, 4, 16), (24, 24, 50400, 2, 0), (32, 32, 69120, 4, 32),
    (48, 48, 125000, 4, 0), (32, 64, 125000, 4, 32), (32, 64, 180000, 4, 0), (32, 32, 1000000, 4, 32),
])
def test_tiles_per_wave(cin, cout, nodes, tiles, ci):
    L = C.CDLL(LIB)
    for f in (L.slbn_conv_ntw, L.slbn_conv_ci):
        f.argtypes = [C.c_int, C.c_int, C.c_long]
    assert (L.slbn_conv_ntw(cin, cout, nodes), L.slbn_conv_ci(cin, cout, nodes)) == (tiles, ci)
