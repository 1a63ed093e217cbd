"""Ladder sums through the shared matrix where device memory is short (needs an MI355X): fewer groups per batch, passes
over the problems left to the LU, and the LU itself where not even one group fits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

GB = 10**9


def _inputs(nb, niv, nq, nw, spoil):
    """Ladder inputs of the tuner's kind; spoil: chi0^-1 of a third of the q-points turned over, which no iteration
    with their mean solves."""
    from dgamore_amd import autotune as A

    inv, gamma, u_r = A._problem(nb, niv, nq, nw, 1)
    if spoil:
        inv = inv * torch.where(torch.arange(nq, device="cuda") % 3 == 0, -1.5, 1.0)
    return inv.contiguous(), gamma, u_r


@pytest.mark.parametrize("leave,nb,niv,nq,nw,precision,spoil", [
    (6.0, 2, 64, 45, 60, 0, True),    # n = 512, 2700 problems: 11.5 GB of LU matrices, 2.6 GB of the shared form
    (6.0, 2, 64, 45, 60, 2, True),
    (2.0, 1, 400, 160, 40, 0, False),  # n = 800: 2.2 GB of matrices and vectors of the shared form's 40 groups
    (2.0, 1, 100, 30, 1200, 0, False),  # n = 200: 3.8 GB of matrices of 1200 groups
])
def test_short_of_memory(leave, nb, niv, nq, nw, precision, spoil, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import kernels as K

    print(f"[gpu-case] shared ladder, {leave} GB free, n={2 * niv * nb * nb} problems={nq * nw} precision={precision}", flush=True)
    ops = _inputs(nb, niv, nq, nw, spoil)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    out_bytes = 16 * ops[0].numel() + (1 << 26)
    free = torch.cuda.mem_get_info()[0] - out_bytes - int(leave * GB)
    fill = torch.empty(max(free, 1), dtype=torch.uint8, device="cuda")
    monkeypatch.setenv("DGAMI_LADDER_SHARED", "1")
    try:
        out, info = K.ladder_solve_sum(*ops, None, 1.0, precision, check_info=False)
        torch.cuda.synchronize()
    finally:
        del fill
        torch.cuda.empty_cache()
    assert not info.any()
    pick = torch.arange(0, nw, max(1, nw // 4), device="cuda")  # the LU of some frequencies
    monkeypatch.setenv("DGAMI_LADDER_SHARED", "0")
    ref, _ = K.ladder_solve_sum(ops[0][pick].contiguous(), ops[1][:, pick].contiguous(), ops[2], None, 1.0)
    err = float((out[:, pick] - ref).abs().max() / ref.abs().max())
    assert err < 1e-11, err
