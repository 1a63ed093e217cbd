"""A batch whose last model cannot be served (needs an MI355X): the call fails, and what the other models' streams
were given is finished before whatever the caller queues next on its own stream."""
import pytest

from tests.conftest import ladder_case

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def test_a_refused_workspace_leaves_no_error_behind():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from dgamore_amd import _lib
    from dgamore_amd import kernels as K

    print("[gpu-case] workspace of a terabyte, then ordinary work", flush=True)
    x = torch.ones(4, dtype=torch.complex128, device="cuda")
    with pytest.raises(RuntimeError):  # refused before anything is launched: the operands are not read
        _lib.call("dgami_dc_kernel", 1 << 26, 2, 64, 8, 8, 1.0, K._p(x), K._p(x), K._p(x), K._p(x), K._stream())
    y = x + 1.0
    out = K.fft_grid(y.reshape(1, 4).clone(), (4, 1, 1), -1)
    torch.cuda.synchronize()
    assert complex(out[0, 0]) == 8.0 and complex(y[0]) == 2.0


def test_streams_are_joined_when_a_model_fails(monkeypatch):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import ctypes

    from dgamore_amd import _lib
    from dgamore_amd import kernels as K

    monkeypatch.setenv("DGAMI_LADDER_SHARED", "1")
    monkeypatch.setenv("DGAMI_LADDER_STREAMS", "2")
    print("[gpu-case] batch of two shared-form models and three that are refused", flush=True)
    nb, niv, nw, nq = 1, 60, 61, 900
    chi0_inv, gamma, u, _, beta = ladder_case(nb, niv, nw - 1, 6, seed=2, with_v=False)
    ci = K.ref4_to_qf(K.to_dev(chi0_inv)).repeat(1, 1, 1, nq // 6).contiguous()
    g, um = K.vertex_to_cmp(K.to_dev(gamma))[None].contiguous(), K.orb_to_m(K.to_dev(u))[None].contiguous()
    ref, _ = K.ladder_solve_sum(ci, g, um, None, beta)
    # one shared-form model per stream; three more, register-kernel models of 2^30 - 1 problems each, are refused
    # together after that, before any of them is launched; the caller's stream copies the others' results next
    outs = [torch.zeros_like(ref) for _ in range(2)]
    infos = [torch.zeros((1, nw, nq), dtype=torch.int32, device="cuda") for _ in range(2)]
    table = (_lib.LadderModel * 5)()
    for m in range(5):
        k, big = min(m, 1), m >= 2
        table[m] = _lib.LadderModel(1, 1 if big else nq, nb, (1 << 30) - 1 if big else nw, 1 if big else niv, beta,
                                    K._p(ci), K._p(g), K._p(um), None, K._p(outs[k]), K._p(infos[k], torch.int32))
    with pytest.raises(ValueError, match="too many problems in one launch"):
        _lib.call("dgami_ladder_solve_sum_multi", 5, ctypes.addressof(table), K._stream())
    copies = [o.clone() for o in outs]
    torch.cuda.current_stream().synchronize()
    for c in copies:
        assert float((c - ref).abs().max() / ref.abs().max()) < 1e-12
