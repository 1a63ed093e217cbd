"""Which form a ladder call takes by itself (needs an MI355X), on either side of the lines of the rule: the two forms'
results differ in their last bits, and each is the same from run to run."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nb,niv,precision,nq,nw,shared", [
    (1, 15, 0, 64, 21, False), (1, 15, 0, 64, 22, True),     # n = 30, 30000 / 11 = 2728 problems
    (1, 20, 0, 45, 20, False), (1, 20, 0, 45, 21, True),     # n = 40, 27000 / 14.3 = 1884
    (1, 48, 0, 40, 13, False), (1, 48, 0, 40, 14, True),     # n = 96, 35000 / 33 = 1061
    (1, 70, 0, 31, 20, False), (1, 70, 0, 31, 21, True),     # n = 140, 60000 / 47.7 = 1259
    (2, 8, 0, 45, 15, False), (2, 8, 0, 45, 16, True),       # n = 64, 9000 / 6.33 = 1422
    (2, 12, 2, 30, 24, False), (2, 12, 2, 30, 26, True),     # n = 96, 13500 / 9 = 1500, also in the mixed forms
    (2, 27, 0, 40, 19, False), (2, 27, 0, 40, 20, True),     # n = 216, 30000 / 19 = 1579
    (2, 33, 0, 64, 22, False), (2, 33, 0, 64, 23, True),     # n = 264, 65000 / 23 = 2827
    (2, 36, 2, 45, 19, False), (2, 36, 2, 45, 21, True),     # n = 288, 45000 / 25 = 1800
    (2, 8, 0, 15, 60, False),                                # 15 q-points are too few
    (3, 20, 0, 64, 60, False),                               # n = 360, T = 9: ratio 14.3
])
def test_form_of_a_call(nb, niv, precision, nq, nw, shared, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import autotune as A
    from dgamore_amd import kernels as K

    print(f"[gpu-case] form of a call: nb={nb} niv={niv} precision={precision} {2 * nq * nw} problems", flush=True)
    A.clear()
    inv, gamma, u_r = A._problem(nb, niv, nq, nw, 2)
    outs = {}
    for form in ("", "0", "1"):
        monkeypatch.setenv("DGAMI_LADDER_SHARED", form)
        outs[form] = K.ladder_solve_sum(inv, gamma, u_r, None, 1.0, precision, check_info=False)[0]
    assert not torch.equal(outs["0"], outs["1"])
    assert torch.equal(outs[""], outs["1" if shared else "0"])
