"""Double-counting kernel at the edges of the product's 64 x 64 x 8 tiles and for every orbital number's
operand form (one orbital: chi0 itself; two to four: a thread's registers; more: the general one).

Sums of at most 150 products in 64 bits: the relative 2-norm error stays below 1e-13.
"""
import numpy as np
import pytest
import torch

from oracle import dga_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,niv_core,niv_shell,nq", [(1, 1, 0, 1), (1, 33, 2, 70), (1, 32, 0, 64), (2, 9, 3, 17),
                                                      (3, 4, 1, 15), (4, 2, 1, 5), (5, 1, 0, 3)])
def test_dc_kernel_edges(nb, niv_core, niv_shell, nq):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import kernels as K

    rng = np.random.default_rng(nb * 100 + nq)
    nw, beta, nvf = 2, 9.0, 2 * (niv_core + niv_shell)

    def cplx(*shape):
        return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)

    chi0, f, u = cplx(nq, nb, nb, nb, nb, nw, nvf), cplx(nb, nb, nb, nb, nw, nvf, nvf), cplx(nb, nb, nb, nb)
    ref = -O.dc_kernel(f, chi0, u, beta, niv_core)
    got = K.qf_to_ref4(K.dc_kernel(K.ref4_to_qf(K.to_dev(chi0)), K.to_dev(u), K.to_dev(f), nb, niv_core, beta), nb)
    got = got.cpu().numpy()
    assert np.linalg.norm(got - ref) < 1e-13 * np.linalg.norm(ref)
