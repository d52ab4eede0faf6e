"""The test that decides whether a wavefront's windows fit its LDS box in the
baseline-layout degridding (csrc/blbox.h), compiled for the host."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    'crocodile_amd', 'csrc')


@pytest.fixture(scope='module')
def box(tmp_path_factory):
    d = tmp_path_factory.mktemp('blbox')
    src, lib = str(d / 'box.cpp'), str(d / 'box.so')
    with open(src, 'w') as f:
        f.write('#include "blbox.h"\n'
                'extern "C" int cells() { return BL_BOX; }\n'
                'extern "C" int fits(int bw, int bh) { return bl_box_fits(bw, bh); }\n')
    subprocess.check_call(['g++', '-std=c++17', '-shared', '-fPIC', '-I', CSRC, src, '-o', lib])
    return ctypes.CDLL(lib)


EDGES = [1, 2, 16, 23, 24, 25, 599, 600, 601, 1000, 23170, 46340, 46341, 46342, 50000, 65535,
         65536, 65552]


@pytest.mark.parametrize('bh', EDGES)
def test_box_holds_what_it_accepts(box, bh):
    """Against the product in Python's integers, up to the whole grid."""
    for bw in EDGES + [1073741824 // bh, 2147483647 // bh, 4294967296 // bh]:
        bw = min(bw, 65552)
        assert bool(box.fits(bw, bh)) == (bh * (bw | 1) <= box.cells()), (bw, bh)
