"""Displacement over timeslices in chunks: 10^3 sites run all path lengths of five
timeslices (1250 workgroups) before the sixth.  Bar: as for the other
displacement tests, FP64 1e-12, mixed 1e-6."""
import numpy as np
import pytest

import easydistillation_amd as ed
from easydistillation_amd import synthetic as S
from oracle import elemental_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("Lt", [5, 6])
def test_chunk_of_five_timeslices(mode, Lt):
    latt, Ne, dist, moms = [10, 10, 10, Lt], 9, 3, S.unit_momenta()
    U, V = S.make_inputs_np(latt, Ne, "haar", seed=Lt)
    g = ed.DisplacementElementalGenerator(latt, None, None, dist, moms, Ne=Ne, mode=mode)
    g.load_arrays(U, V)
    E = g.calc_all()
    ref = O.displacement_elemental(V, U, latt, dist, moms)
    assert np.abs(E - ref).max() <= (1e-12 if mode == "fp64" else 1e-6) * np.abs(ref).max()
