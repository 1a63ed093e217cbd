"""Element counts beyond 2^31 and launches beyond 2^32 work-items (needs an MI355X with 110 GB free): the block
algebra of one orbital on inputs that are products of a frequency and a momentum factor, compared on slices at
the ends and around element 2^31. One product each: 1e-14 covers its few roundings.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

C128 = torch.complex128


@pytest.fixture(scope="module")
def K():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    if torch.cuda.mem_get_info()[0] < 115e9:
        pytest.skip("needs 115 GB of free device memory")
    from dgamore_amd import kernels

    yield kernels
    torch.cuda.empty_cache()


def outer(v, q):
    """[1][1][v][q] of products."""
    x = torch.empty((1, 1, len(v), len(q)), dtype=C128, device="cuda")
    torch.mul(v[:, None], q[None, :], out=x[0, 0])
    return x


def factor(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.view_as_complex(1.0 + 0.3 * torch.randn((n, 2), dtype=torch.float64, device="cuda", generator=g))


def test_vrg_and_kernel_beyond_2_31_elements(K):
    nv, nq = 2048, (1 << 20) + 3
    print(f"[gpu-case] vrg and kernel_r with {nv * nq} elements", flush=True)
    fv, fq = factor(nv, 1), factor(nq, 2)
    x = outer(fv, fq)
    one = torch.ones((1, 1, nq), dtype=C128, device="cuda")
    u = torch.full((1,), 0.25, dtype=C128, device="cuda")
    # chi = ((sum_v x / beta + 0)^-1 + u)^-1
    vrg, chi = K.vrg_chi_phys(x, x, one, one, u, None, 1, 2.0)
    ker = K.kernel_r(vrg, chi, u, None, 1, "magn", 3.0)
    torch.cuda.synchronize()
    for v in (0, 1, nv // 2, nv - 2, nv - 1):  # row 2047 holds element 2^31
        ref = 2.0 * (fv[v] * fq) ** 2
        assert float((vrg[0, 0, v] - ref).abs().max() / ref.abs().max()) < 1e-14, v
        got = 3.0 * 0.25 * (ref - 0.25 * ref * chi[0, 0] - 2.0 / 3.0)
        assert float((ker[0, 0, v] - got).abs().max() / got.abs().max()) < 1e-13, v
    total = fv.sum() * fq / 2.0
    ref = total / (1.0 + 0.25 * total)
    assert float((chi[0, 0] - ref).abs().max() / ref.abs().max()) < 1e-12
