"""Where the block-tridiagonal kernels read a system's super-diagonals (spitfire_amd/csrc/gf_btd_index.h), on the host: the
LAPACK-format solve loads them ahead for every block, also for those that have none."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope='module')
def index(tmp_path_factory):
    so = str(tmp_path_factory.mktemp('btd_index') / 'libindex.so')
    subprocess.run(['g++', '-O1', '-std=c++17', '-shared', '-fPIC', '-o', so,
                    os.path.join(HERE, 'native', 'btd_index_host.cpp')], check=True)
    lib = ctypes.CDLL(so)
    lib.btd_values_host.restype = lib.btd_sup_host.restype = ctypes.c_long
    return lib


@pytest.mark.parametrize('bs', [1, 2, 53, 64])
@pytest.mark.parametrize('nb', [1, 2, 3, 4, 5, 126, 40000])
def test_super_diagonals_are_read_within_the_system(index, nb, bs):
    """Every row that a sweep over the blocks, two at a time and one row ahead, can ask for: in range of the system's values (a
    system may be the last in its buffer), and the row itself wherever there is one."""
    size = nb * bs * bs + 2 * (nb - 1) * bs
    assert index.btd_values_host(nb, bs) == size
    for i in (-2, -1, 0, 1, 2, nb // 2, nb - 3, nb - 2, nb - 1, nb):
        at = index.btd_sup_host(nb, bs, i)
        assert 0 <= at and at + bs <= size
        if 0 <= i < nb - 1:
            assert at == size - (nb - 1 - i) * bs
