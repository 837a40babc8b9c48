"""The list-build driver where cells hold a few particles, entry for entry against the oracle's rows: ragged
cell grids, few cells along an axis, empty and crowded regions, types, exclusions and rows that overflow. The
driver builds by the cell form; the column form (csrc/tile.hip) is tested in test_gpu_columns.py."""

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def H():
    from hoomd_amd import _lib
    assert _lib.lib().hm_device_count() > 0
    return _lib


def box_fluid(N, L, seed):
    L = np.asarray(L, float)
    return np.random.default_rng(seed).uniform(-L / 2, L / 2, (N, 3)), L


def same_rows(got, ref):
    nl, nn, cond = got
    onl, onn = ref
    assert cond[3] == 0
    assert (nn == onn).all()
    k = np.arange(min(nl.shape[1], onl.shape[1]))
    live = k[None, :] < nn[:, None]
    assert np.array_equal(nl[:, :len(k)][live], onl[:, :len(k)][live])
    assert (nl[~(np.arange(nl.shape[1])[None, :] < nn[:, None])] == 0xffffffff).all()


WCA = 2.0 ** (1.0 / 6.0)


@pytest.mark.parametrize("N,L,rcut,buff", [
    (32768, (33.5, 33.6, 33.7), WCA, 0.4),   # 22 cells per axis, 3.1 particles each
    (33333, (6.2, 100.0, 100.0), WCA, 0.4),  # 4 cells along x
    (33001, (150.0, 15.0, 6.9), WCA, 0.4),   # 4 cells along z, 9 along y
    (36001, (30.0, 91.0, 90.0), 2.5, 0.3),   # 10 x 32 x 32 cells
    (36000, (50.0, 51.0, 52.0), 2.5, 0.4),   # 7 particles a cell: 8 lanes per particle
    (40001, (60.0, 61.0, 62.0), WCA, 0.2),   # most cells empty
    (250000, (66.0, 64.0, 70.0), WCA, 0.4),  # columns of several cells
])
def test_rows_equal_oracle(H, N, L, rcut, buff):
    from gpu_helpers import nlist
    pos, L = box_fluid(N, L, N)
    same_rows(nlist(pos, L, rcut, buff), O.nlist_binned(O.Box(*L), pos, rcut, buff, full=True))


def test_crowded_half_of_the_box(H):
    """All particles in half of the box: twice the mean density."""
    from gpu_helpers import nlist
    pos, L = box_fluid(33000, (66.0, 60.0, 62.0), 3)
    pos[:, 0] = pos[:, 0] / 2 + L[0] / 4
    pos[pos[:, 0] >= L[0] / 2, 0] = 0.0
    same_rows(nlist(pos, L, 2.5, 0.4, nmax=160),
              O.nlist_binned(O.Box(*L), pos, 2.5, 0.4, full=True))


def test_types_and_exclusions(H):
    from gpu_helpers import nlist
    N = 33000
    pos, L = box_fluid(N, (49.0, 50.0, 51.0), 5)
    types = (np.arange(N) % 3).astype(np.uint32)
    rc = np.array([[2.5, 1.2, 2.0], [1.2, 0.0, 1.7], [2.0, 1.7, 2.2]])
    same_rows(nlist(pos, L, rc, 0.3, types=types, ntypes=3),
              O.nlist_binned(O.Box(*L), pos, rc, 0.3, full=True, types=types, ntypes=3))
    excl = [[(i + 1) % N, (i - 1) % N, (i + 700) % N, (i - 700) % N] for i in range(N)]
    same_rows(nlist(pos, L, 2.5, 0.4, excl=excl),
              O.nlist_binned(O.Box(*L), pos, 2.5, 0.4, full=True, excl=excl))


def test_overflow_reports_needed_size(H):
    from gpu_helpers import nlist
    pos, L = box_fluid(33000, (50.0, 50.0, 50.0), 8)
    nl, nn, cond = nlist(pos, L, 2.5, 0.4, nmax=8)
    onl, onn = O.nlist_binned(O.Box(*L), pos, 2.5, 0.4, full=True)
    assert cond[3] == onn.max() == nn.max()
    assert (nl == onl[:, :8]).all()
