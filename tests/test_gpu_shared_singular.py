"""Singular ladder matrices whose right-hand sides do not show it, in the shared-matrix form (needs an MI355X): two
equal rows of one orbital pair. Where the LU meets their zero pivot (of real matrices, but for the rounding of a
reciprocal; complex multipliers leave a remainder) the call raises, and so it has to here: info is the LU's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _problem(nb, nv, nq, kind, rng):
    """Real chi0^-1 [1][nb^4][nv][nq], Gamma [1][1][n][n] (beta = 1, U = 0) with two equal rows at q-point 7."""
    T, n, a, b, c = nb * nb, nb * nb * nv, nv // 2, nv - 1, nb * nb - 1
    ci = 0.02 * rng.standard_normal((T, T, nv, nq))
    ci[np.arange(T), np.arange(T)] += 1.0
    if kind == "constant":  # a vertex that does not depend on the frequencies
        g = np.repeat(np.repeat(0.2 / n * rng.standard_normal((T, T)), nv, 0), nv, 1)
    else:
        g = 0.1 / np.sqrt(n) * rng.standard_normal((n, n))
    ra, rb = c * nv + a, c * nv + b
    g[rb] = g[ra]
    if kind == "made up":  # the rows differ in the columns a and b, by what chi0^-1 adds there (powers of two: exact)
        for e in range(T):
            ci[c, e, a, 7], ci[c, e, b, 7] = 0.5 ** (1 + e), 0.25 ** (1 + e)
            g[ra, e * nv + a], g[rb, e * nv + a] = 0.25, 0.25 + 0.5 ** (1 + e)
            g[ra, e * nv + b], g[rb, e * nv + b] = 0.125 + 0.25 ** (1 + e), 0.125
    else:
        ci[c, :, a, 7] = ci[c, :, b, 7] = 0.0
    return ci.reshape(1, T * T, nv, nq).astype(complex), g[None, None].astype(complex)


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("kind", ["constant", "rows", "made up"])
@pytest.mark.parametrize("nb,nv", [(1, 4), (1, 20), (1, 66), (1, 130), (1, 160), (1, 300), (2, 4), (2, 10), (2, 40), (2, 70), (3, 30),
                                   (4, 18)])
def test_equal_rows_are_reported(nb, nv, kind, precision, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import kernels as K

    nq = 18
    print(f"[gpu-case] equal rows: {kind} nb={nb} n={nb * nb * nv} precision={precision}", flush=True)
    ci, g = _problem(nb, nv, nq, kind, np.random.default_rng(nb * nv))
    args = (K.to_dev(ci), K.to_dev(g), torch.zeros((1, nb**4), dtype=torch.complex128, device="cuda"), None, 1.0)
    monkeypatch.setenv("DGAMI_LADDER_SHARED", "0")
    ref, info0 = K.ladder_solve_sum(*args, check_info=False)
    monkeypatch.setenv("DGAMI_LADDER_SHARED", "1")
    out, info = K.ladder_solve_sum(*args, precision, check_info=False)
    assert torch.equal(info, info0)
    keep = [q for q in range(nq) if q != 7]
    assert float((out[..., keep] - ref[..., keep]).abs().max() / ref[..., keep].abs().max()) < 1e-11
    if int(info0[0, 0, 7]) > 0:
        with pytest.raises(np.linalg.LinAlgError):
            K.ladder_solve_sum(*args, precision)


@pytest.mark.parametrize("nb,nv", [(1, 40), (2, 40), (1, 300)])
def test_a_constant_vertex_alone_keeps_the_form(nb, nv, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import kernels as K

    rng = np.random.default_rng(nv)
    T = nb * nb
    ci = 1.0 + 0.05 * rng.standard_normal((1, T * T, nv, 18)) * (1.0 + 0.0j)
    ci[0, [e for e in range(T * T) if e // T != e % T]] *= 0.02
    g = np.full((1, 1, T * nv, T * nv), 0.05 / (T * nv), dtype=complex)
    args = (K.to_dev(ci), K.to_dev(g), torch.zeros((1, nb**4), dtype=torch.complex128, device="cuda"), None, 1.0)
    outs = []
    for form in ("0", "1"):
        monkeypatch.setenv("DGAMI_LADDER_SHARED", form)
        outs.append(K.ladder_solve_sum(*args)[0])
    assert not torch.equal(*outs)  # not the LU's bits
    assert float((outs[0] - outs[1]).abs().max() / outs[0].abs().max()) < 1e-12
