"""Block algebra of the ladder with a block row per wavefront, the frequency sums and the in-place block
inverse: element counts off the wavefronts' 64 (and the 256 of one orbital), every orbital number, with
and without V, added to what is there. Blocks of random numbers (conditions of at most a few hundred):
relative errors stay below 1e-12.
"""
import numpy as np
import pytest
import torch

from oracle import dga_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import kernels

    return kernels


def rel(a, b):
    a = a.cpu().numpy()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def cplx(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


SIZES = [(1, 1, 1, 1), (1, 3, 64, 2), (1, 2, 5, 27), (2, 2, 13, 7), (3, 1, 4, 8), (3, 2, 3, 11), (4, 2, 2, 3),
         (4, 1, 5, 17)]  # nb, nw, niv, nq


@pytest.mark.parametrize("with_v", [False, True])
@pytest.mark.parametrize("nb,nw,niv,nq", SIZES)
def test_vrg_chi_phys_kernel_rows(K, nb, nw, niv, nq, with_v):
    rng = np.random.default_rng(nb + 10 * nq)
    beta, box = 7.0, (nq, nb, nb, nb, nb, nw)
    chi0_inv, aux, full, core = cplx(rng, *box, 2 * niv), cplx(rng, *box, 2 * niv), cplx(rng, *box), cplx(rng, *box)
    ur, vr = cplx(rng, nb, nb, nb, nb), cplx(rng, nq, nb, nb, nb, nb) * (1.0 if with_v else 0.0)
    d = [K.ref4_to_qf(K.to_dev(x)) for x in (chi0_inv, aux)] + [K.ref4w_to_qw(K.to_dev(x)) for x in (full, core)]
    du, dv = K.orb_to_m(K.to_dev(ur)), K.orb_to_m(K.to_dev(vr)) if with_v else None
    vrg, chi = K.vrg_chi_phys(*d, du, dv, nb, beta)
    vrg_ref = O.vrg(chi0_inv, aux, beta)
    assert rel(K.qf_to_ref4(vrg, nb), vrg_ref) < 1e-12
    chi_ref = K.qw_to_ref4w(chi, nb).cpu().numpy()
    for ch in ("dens", "magn"):
        ker = K.kernel_r(vrg, chi, du, dv, nb, ch, 3.0)
        assert rel(K.qf_to_ref4(ker, nb), 3.0 * O.kernel_r(vrg_ref, chi_ref, ur, vr, ch)) < 1e-12


@pytest.mark.parametrize("nb,nw,niv,nq", SIZES)
def test_chi0_sums_and_inverse(K, nb, nw, niv, nq):
    rng = np.random.default_rng(3 + nb + 10 * nq)
    beta, shell = 5.0, 2
    chi0 = cplx(rng, nq, nb, nb, nb, nb, nw, 2 * (niv + shell))
    cut = chi0[..., shell:shell + 2 * niv]
    inv, full, core = K.chi0_prepare(K.ref4_to_qf(K.to_dev(chi0)), nb, niv, beta)
    assert rel(K.qf_to_ref4(inv, nb), O.block_invert_vn1(cut)) < 1e-11  # the worst of up to 900 random blocks
    assert rel(K.qw_to_ref4w(full, nb), chi0.sum(-1) / beta**2) < 1e-12
    assert rel(K.qw_to_ref4w(core, nb), cut.sum(-1) / beta**2) < 1e-12


@pytest.mark.parametrize("nb", [1, 2, 3])
def test_inverse_keeps_a_nan_in_its_block(K, nb):
    rng = np.random.default_rng(nb)
    chi0 = K.ref4_to_qf(K.to_dev(cplx(rng, 5, nb, nb, nb, nb, 2, 6)))
    good, _, _ = K.chi0_prepare(chi0, nb, 3, 5.0)
    chi0[1, nb**4 // 2, 4, 3] = complex(float("nan"), 0.0)
    inv, _, _ = K.chi0_prepare(chi0, nb, 3, 5.0)
    assert torch.isnan(inv[1, :, 4, 3].real).any()
    inv[1, :, 4, 3] = good[1, :, 4, 3]
    assert torch.equal(inv, good)
