"""Ladder sums through the q-points' shared matrix (needs an MI355X): against the oracle at the edges of
its tiles and of its rule, with problems that it has to leave to the LU, and captured in a graph."""
import sys

import numpy as np
import pytest

from oracle import dga_oracle as O
from tests.conftest import ladder_case

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def say(msg):
    print(f"[gpu-case] {msg}", flush=True)
    sys.stdout.flush()


@pytest.fixture(autouse=True)
def shared_form(monkeypatch):
    """The form is taken from far more problems on (ladder_shared.hpp); here wherever it can run."""
    monkeypatch.setenv("DGAMI_LADDER_SHARED", "1")


@pytest.fixture(scope="module")
def K():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import kernels

    return kernels


def _case(nb, niv, niw, nq, seed, spread, with_v):
    """Ladder inputs whose chi0^-1 varies over q by `spread` around that of one q."""
    chi0_inv, gamma, u, v, beta = ladder_case(nb, niv, niw, nq, seed, with_v=with_v)
    rng = np.random.default_rng(seed + 1)
    f = 1.0 + spread * (rng.standard_normal(chi0_inv.shape) + 1j * rng.standard_normal(chi0_inv.shape))
    return chi0_inv[:1] * f, gamma, u, 0.1 * v, beta


def _operands(K, chi0_inv, gamma, u, v):
    g = K.vertex_to_cmp(K.to_dev(gamma))[None].contiguous()
    vd = None if v is None else K.orb_to_m(K.to_dev(v))[None].contiguous()
    return K.ref4_to_qf(K.to_dev(chi0_inv)), g, K.orb_to_m(K.to_dev(u))[None].contiguous(), vd


def _rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


@pytest.mark.parametrize("precision", [0, 1, 2])
@pytest.mark.parametrize("nb,niv,niw,nq,with_v", [
    (1, 1, 1, 2, False),     # n = 2, 2 columns
    (1, 8, 40, 33, True),    # n = 16, one wavefront's rows; 123 tiles
    (1, 17, 1, 16, False),   # n = 34, 16 columns
    (2, 4, 1, 17, True),     # n = 32
    (1, 32, 90, 95, False),  # n = 64, 546 tiles: two workgroups per CU
    (1, 35, 2, 65, True),    # n = 70, one column in the second tile, V_r
    (1, 60, 0, 64, False),   # n = 120, exactly four tiles
    (1, 64, 0, 20, True),    # n = 128, the largest of four-wavefront tiles
    (1, 65, 0, 20, False),   # n = 130
    (2, 9, 1, 17, False),    # n = 72, 68 columns: a q-point in both tiles' range
    (2, 14, 1, 16, True),    # n = 112
    (3, 4, 2, 16, False),    # n = 72, 9 right-hand sides that cross the tiles
    (3, 9, 0, 23, True),     # n = 162
    (4, 3, 0, 17, True),     # n = 96, 16 right-hand sides
    (4, 8, 0, 17, False),    # n = 256, the largest of the tiles
    (1, 129, 0, 65, True),   # n = 258, the large form
    (2, 33, 0, 19, False),   # n = 264
    (3, 15, 1, 16, True),    # n = 270
])
def test_shared_ladder_matches_oracle(K, nb, niv, niw, nq, with_v, precision):
    say(f"shared ladder nb={nb} niv={niv} niw={niw} nq={nq} n={nb * nb * 2 * niv} V={with_v} precision={precision}")
    chi0_inv, gamma, u, v, beta = _case(nb, niv, niw, nq, 7 * nb + niv, 0.03, with_v)
    ref = O.ladder_sum_solve(chi0_inv, gamma, u, v, beta)
    out, info = K.ladder_solve_sum(*_operands(K, chi0_inv, gamma, u, v if with_v else None), beta, precision)
    torch.cuda.synchronize()
    assert int(info.abs().sum()) == 0
    # complex128: the oracle's own LU differs from the exact solution by cond * 2^-53 (cond <= 1e4 here)
    assert _rel(K.qf_to_ref4(out[0], nb).cpu().numpy(), ref) < (1e-10 if precision == 0 else 1e-8)


@pytest.mark.parametrize("precision", [1, 2])
@pytest.mark.parametrize("spread", [0.03, 0.15])
@pytest.mark.parametrize("nb,niv,niw,nq,with_v", [
    (1, 129, 0, 65, False),  # n = 258, one column in the second tile
    (1, 129, 0, 65, True),
    (2, 33, 1, 19, True),    # n = 264
    (3, 16, 0, 17, False),   # n = 288
    (4, 9, 0, 17, True),     # n = 288, 272 columns
    (3, 40, 0, 16, False),   # n = 720
])
def test_complex64_basis_matches_the_fp64_form(K, nb, niv, niw, nq, with_v, spread, precision):
    """The mixed forms above n = 256 iterate in complex64 on FP64 residuals: |X| to 1e-14 times the norm
    of the inverse of 1 + P D(q), at most ten here, where both forms converge."""
    say(f"complex64 basis nb={nb} niv={niv} nq={nq} n={nb * nb * 2 * niv} V={with_v} spread={spread}")
    chi0_inv, gamma, u, v, beta = _case(nb, niv, niw, nq, 7 * nb + niv, spread, with_v)
    ops = _operands(K, chi0_inv, gamma, u, v if with_v else None)
    ref, info0 = K.ladder_solve_sum(*ops, beta)
    out, info = K.ladder_solve_sum(*ops, beta, precision)
    torch.cuda.synchronize()
    assert not info.any() and not info0.any()
    assert float((out - ref).abs().max() / ref.abs().max()) < 1e-11


@pytest.mark.parametrize("precision", [0, 2])
@pytest.mark.parametrize("niv", [80, 130])  # n = 160: tiles; 260: the large form
def test_singular_leading_block_takes_the_lu(K, niv, precision):
    """Mean matrices that are regular but whose leading 64 x 64 block vanishes: the block-wise inversion
    pivots inside its blocks only and has no inverse to offer."""
    nq = 18
    say(f"shared ladder, vanishing leading block: n={2 * niv} precision={precision}")
    chi0_inv, gamma, u, v, beta = _case(1, niv, 0, nq, 3, 0.01, False)
    mean = chi0_inv.mean(axis=0)[0, 0, 0, 0]  # [w, v]
    block = u.reshape(()) * np.ones((64, 64)) - beta**2 * np.stack([np.diag(m[:64]) for m in mean])
    gamma = gamma.copy()
    gamma[0, 0, 0, 0, :, :64, :64] = block
    ref = O.ladder_sum_solve(chi0_inv, gamma, u, v, beta)
    out, info = K.ladder_solve_sum(*_operands(K, chi0_inv, gamma, u, None), beta, precision)
    torch.cuda.synchronize()
    assert not info.any()
    # (no error bound below the conditioning of these matrices is known in advance)
    assert _rel(K.qf_to_ref4(out[0], 1).cpu().numpy(), ref) < (1e-8 if precision == 0 else 1e-6)


@pytest.mark.parametrize("nb,niv,nq", [(1, 40, 20), (2, 20, 18), (2, 33, 16)])  # n = 80: column kernel; 160, 264: blocked LU
def test_unconverged_problems_take_the_lu(K, nb, niv, nq):
    """chi0^-1 that differs between the q-points by more than its mean: the iteration does not converge
    and every problem is solved by the LU; one singular matrix is reported as the LU reports it."""
    say(f"shared ladder, unrelated q-points: nb={nb} niv={niv} nq={nq} n={nb * nb * 2 * niv}")
    chi0_inv, gamma, u, v, beta = ladder_case(nb, niv, 1, nq, seed=5, with_v=False)
    scale = np.where(np.arange(nq) % 2 == 0, 1.0, -1.3)[:, None, None, None, None, None, None]
    chi0_inv = chi0_inv * scale
    ref = O.ladder_sum_solve(chi0_inv, gamma, u, v, beta)
    ops = _operands(K, chi0_inv, gamma, u, None)
    out, info = K.ladder_solve_sum(*ops, beta)
    torch.cuda.synchronize()
    assert int(info.abs().sum()) == 0
    assert _rel(K.qf_to_ref4(out[0], nb).cpu().numpy(), ref) < 1e-10
    bad = ops[0].clone()
    bad[1, 0, 3, 2] = complex(float("nan"), 0.0)
    out2, info2 = K.ladder_solve_sum(bad, *ops[1:], beta, check_info=False)
    torch.cuda.synchronize()
    info2 = info2.cpu().numpy()
    assert info2[0, 1, 2] != 0 and np.count_nonzero(info2) == 1
    keep = [q for q in range(nq) if q != 2]
    assert float((out2[..., keep] - out[..., keep]).abs().max() / out.abs().max()) < 1e-12
    with pytest.raises(np.linalg.LinAlgError):
        K.ladder_solve_sum(bad, *ops[1:], beta)


@pytest.mark.parametrize("precision", [0, 2])
def test_captured_shared_step_replays_match_eager(K, precision):
    from dgamore_amd import synthetic as S
    from dgamore_amd.pipeline import SDEPipeline

    say(f"graph capture of an SDE step with the shared ladder: 1 band 10x10 niw=2 niv=36 (n=72), precision {precision}")
    m = S.make_model(0, nk=(10, 10, 1), niw=2, niv=36)
    pipe = SDEPipeline(m, precision=precision, mixing=0.3)
    pipe.capture()
    for it in range(3):
        inp = pipe.graph_sigma.clone()
        out, info = pipe.replay().clone(), pipe.last_info.clone()
        torch.cuda.synchronize()
        ref = pipe.step(inp, m.mu)
        torch.cuda.synchronize()
        assert not info.any()
        assert float((out - ref).abs().max() / ref.abs().max()) < 1e-13, it
        pipe.graph_sigma.copy_(out)
        torch.cuda.synchronize()


@pytest.mark.parametrize("precision", [0, 2])
def test_batch_spreads_its_models_over_streams(K, precision):
    """Models of a batch in the shared form on the caller's and the extra streams, beside one for the LU
    (n above the form's one-launch sizes) and one that does not converge: each as in a call of its own."""
    say(f"batch of shared-form models, precision {precision}")
    shapes = [(1, 20, 2, 17), (2, 8, 1, 16), (1, 36, 0, 33), (2, 20, 0, 16), (1, 10, 3, 18)]
    models = []
    for k, (nb, niv, niw, nq) in enumerate(shapes):
        chi0_inv, gamma, u, _, beta = _case(nb, niv, niw, nq, 11 + k, 0.03 if k < 4 else 3.0, False)
        models.append((*_operands(K, chi0_inv, gamma, u, None), beta))
    for _ in range(2):
        outs = K.ladder_solve_sum_multi(models, precision=precision)
        torch.cuda.synchronize()
        for m, o in zip(models, outs):
            ref, info = K.ladder_solve_sum(*m, precision)
            assert not info.any()
            assert float((o[0] - ref).abs().max() / ref.abs().max()) < (1e-13 if precision == 0 else 1e-9)
