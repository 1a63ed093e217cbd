"""The complex64 basis of the shared-matrix ladder where it loses its norms (needs an MI355X): D(q) close to a
multiple of the mean matrix, so that the remainder of an orthogonalisation is below the rounding of the basis.

A column is done at a residual |P (B - A X)| of at most 2e-14 |X| as the stored vectors give it; the rounding of
the products adds 2^-16 |P D| |y| with |y| <= 1e-9 |X| and |P D| <= 1.2 here: 2e-14. 1e-13 covers both.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("precision", [1, 2])
@pytest.mark.parametrize("rho", [1.0, 2.0, 4.0])
def test_residual_where_the_basis_degenerates(rho, precision, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import kernels as K

    monkeypatch.setenv("DGAMI_LADDER_SHARED", "1")
    n, pairs = 384, 150  # 384: single precision rounds 1 / sqrt(n) up, which all elements of a vector may hold
    print(f"[gpu-case] degenerate complex64 basis rho={rho} precision={precision}", flush=True)
    rng = np.random.default_rng(int(rho))
    s = np.where(np.arange(n) % 2 == 0, 1.0, -1.0)
    gamma = (1.0 / rho - 1.0) * np.outer(s, s) / n  # A0 = 1 + gamma: 1 on all vectors but s, 1 / rho there
    c = rng.uniform(0.3, 0.6, pairs) / max(rho / 2.0, 1.0)
    d = np.exp(rng.uniform(np.log(1e-5), np.log(2e-4), pairs))
    c, d = np.stack([c, -c], 1).ravel(), np.stack([d, -d], 1).ravel()
    ci = 1.0 + c[None, :] + d[None, :] * s[:, None]
    out, info = K.ladder_solve_sum(K.to_dev(ci[None, None]), K.to_dev(gamma[None, None]),
                                   torch.zeros((1, 1), dtype=torch.complex128, device="cuda"), None, 1.0, precision)
    torch.cuda.synchronize()
    assert not info.any()
    x = out[0, 0, 0].cpu().numpy()  # [v][q]
    a0 = np.diag(ci.mean(axis=1)) + gamma
    left = np.linalg.solve(a0, 1.0 - ci * x - gamma @ x)
    worst = float((np.linalg.norm(left, axis=0) / np.linalg.norm(x, axis=0)).max())
    print(f"worst residual {worst:.2e}", flush=True)
    assert worst < 1e-13
