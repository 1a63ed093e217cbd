"""Ladder sums through the shared matrix in several batches of groups, whose last is shorter (needs an MI355X with
70 GB free): more groups than 24 GiB hold, compared with calls for some frequencies alone, which are one batch.
Some problems of every batch do not converge and go to the LU, whose updates walk their list 64 at a time."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nb,niv,nq,nw,precision", [
    (1, 128, 16, 11000, 0),    # n = 256, tiles: 4.7 MB of matrices per group, three batches of up to 5440
    (1, 129, 20000, 50, 0),    # n = 258, large form: 1.2 GB of vectors per group, batches of 20, 20 and 10
    (1, 129, 20000, 90, 2),    # the same in complex64: 0.7 GB
])
def test_batches_of_groups(nb, niv, nq, nw, precision, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 70e9:
        pytest.skip("needs 70 GB of free device memory")
    from dgamore_amd import autotune as A
    from dgamore_amd import kernels as K

    print(f"[gpu-case] shared ladder in batches: n={2 * niv} nq={nq} nw={nw} precision={precision}", flush=True)
    monkeypatch.setenv("DGAMI_LADDER_SHARED", "1")
    inv, gamma, u_r = A._problem(nb, niv, nq, nw, 1)
    pick = torch.linspace(0, nw - 1, 9).long().cuda()
    turned = torch.arange(0, nq, max(2, nq // 40), device="cuda")
    sub = inv[pick]
    sub[..., turned] *= -1.5  # no iteration with the mean solves these q-points
    inv[pick] = sub
    out, info = K.ladder_solve_sum(inv, gamma, u_r, None, 1.0, precision, check_info=False)
    torch.cuda.synchronize()
    assert not info.any()
    del inv
    torch.cuda.empty_cache()
    for i, w in enumerate(pick.tolist()):
        ref, _ = K.ladder_solve_sum(sub[i:i + 1].contiguous(), gamma[:, w:w + 1].contiguous(), u_r, None, 1.0, precision,
                                    check_info=False)
        assert float((out[:, w:w + 1] - ref).abs().max() / ref.abs().max()) < 1e-12, w
    monkeypatch.setenv("DGAMI_LADDER_SHARED", "0")
    w, q = int(pick[-1]), torch.arange(0, nq, max(1, nq // 50), device="cuda")
    ref, _ = K.ladder_solve_sum(sub[-1:, ..., q].contiguous(), gamma[:, w:w + 1].contiguous(), u_r, None, 1.0)
    assert float((out[:, w:w + 1][..., q] - ref).abs().max() / ref.abs().max()) < 1e-11
    del out, info, gamma, sub
    torch.cuda.empty_cache()
