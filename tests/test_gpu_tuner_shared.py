"""The autotuner where the q-points' shared matrix would serve its batch (needs an MI355X): what it times, compares and
stores are LU kernels, and the form of later calls does not change."""
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("nb,niv,nq,nw,precision", [(1, 20, 64, 20, 0), (2, 8, 40, 20, 0), (3, 45, 40, 16, 2)])
def test_tuner_times_the_lu(nb, niv, nq, nw, precision, tmp_path, monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import autotune as A
    from dgamore_amd import kernels as K

    n, T = nb * nb * 2 * niv, nb * nb
    print(f"[gpu-case] tuner with {2 * nq * nw} problems of n={n}, precision {precision}", flush=True)
    monkeypatch.setenv(A.CACHE_ENV, str(tmp_path / "tune.json"))
    solve, seen = K.ladder_solve_sum, {}

    def recorded(inv, gamma, u_r, *args, **kw):
        out = solve(inv, gamma, u_r, *args, **kw)
        seen.setdefault(A.get_choice(n, T, precision), ((inv, gamma, u_r), out[0]))
        return out

    A.clear()
    try:
        monkeypatch.setenv("DGAMI_LADDER_SHARED", "1")
        monkeypatch.setattr(K, "ladder_solve_sum", recorded)
        r = A.tune_ladder(nb, niv, nq, nw, precision=precision, reps=1)
        monkeypatch.setattr(K, "ladder_solve_sum", solve)
        assert r["source"] == "timed" and set(seen) == {None, *A.candidates(n, T, precision)}
        inputs = seen[None][0]
        shared, _ = solve(*inputs, None, 1.0, precision)  # of this thread again
        assert not torch.equal(shared, seen[None][1])
        monkeypatch.setenv("DGAMI_LADDER_SHARED", "0")
        for kid, (_, out) in seen.items():
            A.set_choice(n, T, precision, kid)
            assert torch.equal(out, solve(*inputs, None, 1.0, precision)[0]), kid
    finally:
        A.clear()
