"""The contraction adjoint's split into workgroups (16, 8 or 4 rows at 64 sites,
in ranges per XCD): several row groups with a ragged last one, sites past a
multiple of 64, counts that do not divide by eight, and one, two and more split
terms with 4, 8 and more momentum groups, against FP64 torch autograd.

Bar: as for the adjoint's other tests, 1e-11 normwise -- 1e5 roundings of FP64,
for sums of at most 8 x 3 x 49 x 27 terms.
"""
import numpy as np
import pytest
import torch

from easydistillation_amd import synthetic as S
from easydistillation_amd.autograd import ElementalEngine
from oracle import elemental_oracle as O
from oracle import elemental_torch as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "latt,Ne,nn,moms",
    [
        ([5, 3, 7, 3], 33, 0, S.unit_momenta()),  # 48 rows, one split term
        ([5, 3, 7, 3], 33, 1, S.momenta_by_norm(2)),  # two terms, more than eight groups
        ([4, 4, 4, 1], 16, 1, S.unit_momenta()),  # one row group, 64 sites: one workgroup
        ([3, 5, 9, 2], 49, 2, [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 1, 0), (0, 1, 1)]),  # eight groups
    ],
)
def test_row_and_site_groups(latt, Ne, nn, moms):
    rng = np.random.default_rng(Ne + nn)
    U = S.gauge_np(rng, latt, "haar")
    V = S.eigvecs_np(rng, latt, Ne).astype(np.complex128)
    D = O.num_derivative(nn)
    G = torch.from_numpy(rng.normal(size=(latt[3], D, len(moms), Ne, Ne, 2))).double()
    G = torch.view_as_complex(G)
    Ut, Vt = torch.from_numpy(U).requires_grad_(), torch.from_numpy(V).requires_grad_()
    want = torch.autograd.grad((G.conj() * T.elemental(Vt, Ut, latt, nn, moms, None)).real.sum(), [Ut, Vt],
                               allow_unused=True)
    Ud, Vd = Ut.detach().cuda(), Vt.detach().cuda()
    eng = ElementalEngine(latt, Ne, nn, moms, None)
    eng.forward(Ud, Vd)
    got = eng.backward(Ud, Vd, G.cuda())
    for g, w in zip(got, want):
        g = g.cpu()
        if w is None:
            assert g.abs().max() == 0  # no derivatives: E does not depend on U
        else:
            assert (g - w).abs().max() <= 1e-11 * w.abs().max()
