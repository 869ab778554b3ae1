"""The block Laplacian's vectors per thread (1, 4 or 8 by the size of the call):
each form and its last, shorter group of vectors against the call's own result
one vector at a time (the arithmetic of a site is the same: equal to rounding),
and that against the dense oracle."""
import numpy as np
import pytest
import torch

import easydistillation_amd.synthetic as S
from easydistillation_amd.eigen import EigenvectorGenerator
from oracle import eigen_oracle as EO

pytestmark = pytest.mark.gpu


# 16 site blocks of 256 (the last one ragged): 4096 and 8192 pairs lie at 256 and 512 vectors
@pytest.mark.parametrize("nvec", [3, 255, 256, 257, 511, 512, 517])
def test_vectors_per_thread(nvec):
    latt = [15, 17, 16, 2]
    Lx, Ly, Lz, _ = latt
    rng = np.random.default_rng(nvec)
    gen = EigenvectorGenerator(latt, None, 4)
    U = S.gauge_np(rng, latt, "haar")
    gen.load_links(U)
    F = torch.complex(*(torch.randn(nvec, Lz, Ly, Lx, 3, dtype=torch.float64, device="cuda") for _ in range(2)))
    got = gen.laplacian(1, F)
    # |out| <= 12 |F| site by site: 55 rounded terms of size <= |F|
    tol = 64 * np.finfo(float).eps * 12 * F.abs().max().item()
    for v in sorted({0, nvec // 2, nvec - 2, nvec - 1}):
        one = gen.laplacian(1, F[v : v + 1].contiguous())
        assert (got[v] - one[0]).abs().max().item() <= tol
    want = np.moveaxis(EO.laplacian(np.moveaxis(F[-2:].cpu().numpy(), 0, -1), U[:, 1]), -1, 0)
    assert np.abs(got[-2:].cpu().numpy() - want).max() <= tol
