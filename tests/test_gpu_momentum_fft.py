"""Momentum transforms on grids with every radix, axis order and row padding, and what is fused into
them: the bubble's -R product and the self-energy's gather from LDS or from memory.

A transform of N points loses at most a few log2(N) roundings of 2^-53 (relative 2-norm): 1e-14 holds
for every size below; the sums of the bubble and the self-energy are compared at 1e-12.
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
    a = a.cpu().numpy() if isinstance(a, torch.Tensor) else a
    return np.linalg.norm(a - b) / np.linalg.norm(b)


GRIDS = [(1, 1, 1), (1, 1, 2), (3, 1, 1), (1, 5, 1), (6, 1, 1), (2, 8, 1), (9, 1, 10), (12, 15, 1), (5, 6, 8),
         (8, 4, 18), (27, 25, 1), (30, 1, 32), (2, 3, 125), (48, 48, 1), (48, 80, 1), (64, 32, 2), (64, 64, 1),
         (4096, 1, 1)]


@pytest.mark.parametrize("nk", GRIDS)
@pytest.mark.parametrize("sign", [-1, 1])
def test_grid(K, nk, sign):
    rng = np.random.default_rng(int(np.prod(nk)))
    x = rng.standard_normal((3,) + nk) + 1j * rng.standard_normal((3,) + nk)
    ref = np.fft.fftn(x, axes=(1, 2, 3)) if sign < 0 else np.fft.ifftn(x, axes=(1, 2, 3)) * np.prod(nk)
    got = K.fft_grid(K.to_dev(x.reshape(3, -1)), nk, sign, 1.0)
    assert rel(got.reshape((3,) + nk), ref) < 1e-14


@pytest.mark.parametrize("nk", [(4097, 1, 1), (50, 81, 1), (7, 4, 1)])
def test_grid_refused(K, nk):
    x = torch.zeros((1, int(np.prod(nk))), dtype=torch.complex128, device="cuda")
    with pytest.raises(Exception):
        K.fft_grid(x, nk, 1, 1.0)


@pytest.mark.parametrize("nk", [(1, 1, 1), (6, 1, 1), (1, 9, 4), (5, 6, 8), (16, 1, 12)])
def test_bubble(K, nk):
    nb, niw, niv, beta, N = 2, 2, 3, 7.0, int(np.prod(nk))
    rng = np.random.default_rng(N)
    ng = 2 * (niw + niv)
    g = rng.standard_normal(nk + (nb, nb, ng)) + 1j * rng.standard_normal(nk + (nb, nb, ng))
    ind = np.arange(N)[::-1].copy()  # every point, in another order
    ref = O.bubble_fft(g, niw, niv, ind, beta)
    got = K.qf_to_ref4(K.bubble_irrq(K.to_dev(g), nk, niw, niv, beta, K.to_dev(ind, torch.int32)), nb)
    assert rel(got, ref) < 1e-12


@pytest.mark.parametrize("reduced", [True, False])
@pytest.mark.parametrize("nk", [(2, 1, 1), (8, 8, 1), (5, 4, 6), (64, 32, 2)])
def test_sigma(K, nk, reduced):
    nb, niw, niv, beta, N = (1 if np.prod(nk) > 1000 else 2), 2, 3, 6.0, int(np.prod(nk))
    rng = np.random.default_rng(N)
    nq = N // 2 if reduced else N
    inv = rng.integers(0, nq, N)
    shape = (nq,) + (nb,) * 4 + (niw + 1, 2 * niv)
    kern = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    shape = nk + (nb, nb, 2 * (niw + niv + 1))
    g = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    ref = O.sigma_fft(kern, g, inv, beta, niv, niw)
    got = K.sigma_from_kernel(K.ref4_to_qf(K.to_dev(kern)), K.to_dev(inv, torch.int32), K.to_dev(g), nk, niw, beta)
    assert rel(got, ref) < 1e-12


@pytest.mark.parametrize("nq", [2, 5])
def test_sigma_entry_outside_the_list_reads_nan(K, nq):
    nk, niw, niv = (4, 2, 1), 1, 2
    inv = np.arange(8) % nq
    inv[3] = nq
    kern = torch.ones((niw + 1, 1, 2 * niv, nq), dtype=torch.complex128, device="cuda")
    g = torch.ones(nk + (1, 1, 2 * (niw + niv)), dtype=torch.complex128, device="cuda")
    out = K.sigma_from_kernel(kern, K.to_dev(inv, torch.int32), g, nk, niw, 5.0)
    assert torch.isnan(out.real).all()
