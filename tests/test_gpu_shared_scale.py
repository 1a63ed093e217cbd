"""Ladder sums through the shared matrix at the ends of the floating-point range (needs an MI355X).

The matrices are scaled by a power of two, which scales the solution by its inverse without a rounding: the
result has to be that of the unscaled call to 1e-11 (both forms are at 1e-13 or better on these matrices). Columns
whose norms would underflow in the iteration have to go to the LU.
"""
import numpy as np
import pytest

from tests.conftest import ladder_case

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("power", [-600, -300, 60, 300, 500, 565, 900])
@pytest.mark.parametrize("nb,niv,precision", [(1, 20, 0), (2, 9, 0), (1, 70, 0), (1, 130, 0)])
def test_scaled_matrices(nb, niv, precision, power, monkeypatch):
    _compare(nb, niv, precision, power, monkeypatch)


@pytest.mark.parametrize("power", [-130, -70, 60, 100, 120, 125])
@pytest.mark.parametrize("precision", [1, 2])
def test_scaled_matrices_complex64_basis(precision, power, monkeypatch):
    _compare(1, 130, precision, power, monkeypatch)


def _compare(nb, niv, precision, power, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import kernels as K

    monkeypatch.setenv("DGAMI_LADDER_SHARED", "1")
    print(f"[gpu-case] scaled ladder nb={nb} niv={niv} precision={precision} 2^{power}", flush=True)
    chi0_inv, gamma, u, _, beta = ladder_case(nb, niv, 1, 18, seed=nb + niv, with_v=False)
    rng = np.random.default_rng(niv)
    chi0_inv = chi0_inv[:1] * (1.0 + 0.05 * rng.standard_normal(chi0_inv.shape))
    ci = K.ref4_to_qf(K.to_dev(chi0_inv))
    g = K.vertex_to_cmp(K.to_dev(gamma))[None].contiguous()
    um = K.orb_to_m(K.to_dev(u))[None].contiguous()
    ref, _ = K.ladder_solve_sum(ci, g, um, None, beta)
    s = 2.0 ** power
    out, info = K.ladder_solve_sum(ci * s, g * s, um * s, None, beta, precision)
    torch.cuda.synchronize()
    assert not info.any()
    err = float((out * s - ref).abs().max() / ref.abs().max())
    assert err < 1e-11
