"""The ladder's info is read after the rest of a step is queued: items of a mixed solve that failed are
solved again and the step is formed anew, a singular matrix raises and leaves the pipeline as it was."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture
def K(monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import kernels

    return kernels


def _spoil(K, monkeypatch, name, value):
    """The next call of the solve leaves a garbage item with this info."""
    solve, left = getattr(K, name), [1]

    def wrapped(*args, **kw):
        out = solve(*args, **kw)
        if left[0]:
            left[0] = 0
            aux, info = out if name == "ladder_solve_sum" else out[-1]
            aux[1, 2, ..., 3] = float("nan")
            info[1, 2, 3] = value
        return out

    monkeypatch.setattr(K, name, wrapped)


@pytest.mark.parametrize("batch", [False, True])
def test_failed_items_are_solved_again(K, monkeypatch, batch):
    from dgamore_amd import synthetic as S
    from dgamore_amd.pipeline import ModelBatch, SDEPipeline

    models = [S.make_model(k, nk=(8, 8, 1), niw=3, niv=36) for k in range(2)]  # n = 72: a blocked-LU size
    run = ModelBatch(models, precision=1) if batch else SDEPipeline(models[0], precision=1, mixing=0.3)
    ref = run.step()
    _spoil(K, monkeypatch, "ladder_solve_sum_multi" if batch else "ladder_solve_sum", -1)
    got = run.step()
    for a, b in zip(got if batch else [got], ref if batch else [ref]):
        assert float((a - b).abs().max() / b.abs().max()) < 1e-8  # the mixed solve against FP64


@pytest.mark.parametrize("batch", [False, True])
def test_singular_matrix_raises_and_keeps_the_last_step(K, monkeypatch, batch):
    from dgamore_amd import synthetic as S
    from dgamore_amd.pipeline import ModelBatch, SDEPipeline

    models = [S.make_model(k, nk=(8, 8, 1), niw=3, niv=6) for k in range(2)]
    run = ModelBatch(models) if batch else SDEPipeline(models[0], mixing=0.3)
    run.step(keep=True)
    pipes = run.pipes if batch else [run]
    before = [p.last for p in pipes]
    _spoil(K, monkeypatch, "ladder_solve_sum_multi" if batch else "ladder_solve_sum", 4)
    with pytest.raises(np.linalg.LinAlgError):
        run.step(keep=True)
    assert all(p.last is b for p, b in zip(pipes, before))
