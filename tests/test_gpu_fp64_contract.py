"""FP64 contraction at the edges of its tiling: tile groups (one tile, odd and
even tile counts, three- and four-tile groups of up to six row blocks), line
lengths from 1 up, line ranges inside a plane and over several planes, every
slot pattern of the momentum blocks and lists that need several blocks, and
three derivatives (five and more split terms).

Bar: 1e-12 blockwise against the oracle, the FP64 form's own (the oracle and the
kernel each round at 1e-16 per term, over at most 2e3 terms here).
"""

import numpy as np
import pytest

import easydistillation_amd as ed
from easydistillation_amd import synthetic as S
from oracle import elemental_oracle as O

pytestmark = pytest.mark.gpu

LINE_Z = [(0, 0, k) for k in range(-70, 71, 2)]  # more z functions than one block holds
AXES = [(3, 0, 0), (0, -3, 0), (2, 2, 0), (-2, 1, 3), (7, 0, 1), (0, 5, -2), (1, 1, 1), (3, 3, 3), (1, 1, 1)]

CASES = [
    # (latt, Ne, nabla, momenta)
    ([4, 4, 4, 1], 1, 1, S.momenta_by_norm(0)),      # one product, one tile
    ([1, 3, 4, 2], 16, 1, S.momenta_by_norm(1)),     # one site per line
    ([2, 5, 3, 1], 17, 2, S.momenta_by_norm(2)),     # two tiles a side, one three-tile group
    ([5, 4, 3, 1], 48, 2, S.momenta_by_norm(4)),     # three tiles a side
    ([5, 4, 3, 2], 65, 1, S.momenta_by_norm(4)),     # five: last row and column in runs
    ([4, 4, 4, 1], 128, 2, S.momenta_by_norm(1)),    # eight: diagonal blocks share every fourth
    ([4, 6, 3, 1], 136, 1, S.momenta_by_norm(3)),    # nine
    ([3, 4, 5, 2], 20, 1, S.momenta_by_norm(9)),     # two momentum blocks
    ([4, 3, 6, 1], 9, 1, LINE_Z),                    # blocks split over z functions
    ([9, 5, 4, 1], 33, 1, AXES),                     # components past 2, repeats, |n| above L
    ([3, 3, 4, 1], 18, 3, S.momenta_by_norm(2)),     # three derivatives
    ([4, 3, 3, 1], 20, 3, S.momenta_by_norm(9)),
    ([16, 16, 5, 1], 16, 0, S.momenta_by_norm(1)),   # planes in parts
    ([12, 2, 9, 8], 40, 2, S.momenta_by_norm(1)),    # several planes per range
]


@pytest.mark.parametrize("latt,Ne,nabla,moms", CASES)
def test_fp64_contraction_against_oracle(latt, Ne, nabla, moms):
    U, V = S.make_inputs_np(latt, Ne, "haar", seed=7 + Ne)
    ref = O.elemental(V, U, latt, nabla, moms)
    g = ed.ElementalGenerator(latt, None, None, nabla, moms, Ne=Ne)
    g.load_arrays(U, V)
    E = g.calc_all()
    d = np.abs(E - ref).max((0, 3, 4))
    r = np.abs(ref).max((0, 3, 4))
    row = r.max(1, keepdims=True)
    # blocks that vanish by symmetry are measured against their derivative's scale
    assert (d / np.where(r >= 1e-8 * row, r, row)).max() <= 1e-12
    # a timeslice alone gives the same bits as in the batch
    g1 = ed.ElementalGenerator(latt, None, None, nabla, moms, Ne=Ne)
    g1.load_arrays(U, V)
    t = latt[3] - 1
    assert np.array_equal(g1.calc_range(t, 1)[0], E[t])


@pytest.mark.parametrize("latt,Ne", [([3, 3, 3, 1], 1), ([4, 4, 5, 3], 63), ([4, 4, 5, 2], 64), ([5, 7, 9, 2], 65),
                                     ([6, 6, 6, 1], 130), ([16, 16, 16, 1], 70)])
@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
def test_orthonormality_of_uneven_blocks(latt, Ne, dtype):
    """max|V^dag V - 1| over 64 x 64 tiles and ranges of sites, one eigenvector off by 1e-3."""
    rng = np.random.default_rng(Ne)
    V = S.eigvecs_np(rng, latt, Ne)
    V[latt[3] - 1, Ne - 1] *= np.float32(1.001)
    g = ed.ElementalGenerator(latt, None, None, 0, [(0, 0, 0)], Ne=Ne)
    g.load_arrays(S.gauge_np(rng, latt, "unit"), V.astype(dtype))
    W = V.astype(np.complex128).reshape(latt[3], Ne, -1)
    want = max(np.abs(w.conj() @ w.T - np.eye(Ne)).max() for w in W)
    # both sum products of complex64 values in FP64: K terms of at most 1, 1e-16 each
    assert abs(g.context.orthonormality() - want) <= 1e-13
