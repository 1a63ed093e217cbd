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


def test_frequency_sums_of_2_30_momenta(K):
    nq = (1 << 30) + 5
    print(f"[gpu-case] frequency sums over {nq} momenta", flush=True)
    x = torch.empty((1, 1, 2, nq), dtype=C128, device="cuda")
    x[0, 0, 0] = 1.5 + 0.25j
    x[0, 0, 1] = -0.5 + 1.0j
    marks = [0, 63, 64, (1 << 28) - 1, 1 << 28, (1 << 28) + 64, 1 << 30, nq - 1]
    for i, q in enumerate(marks):
        x[0, 0, 0, q] = 10.0 + i
    inv, full, core = K.chi0_prepare(x, 1, 1, 2.0)
    torch.cuda.synchronize()
    del inv, core
    want = torch.full((nq,), (1.0 + 1.25j) / 4.0, dtype=C128, device="cuda")
    for i, q in enumerate(marks):
        want[q] = (9.5 + i + 1.0j) / 4.0
    assert torch.equal(full[0, 0], want)


def test_bubble_of_2_23_slabs_of_4096_points(K):
    nk, niw, niv, beta = (64, 64, 1), 2047, 2048, 2.0
    print("[gpu-case] bubble of 2^23 slabs of 64x64", flush=True)
    ng = niw + niv
    gen = torch.Generator(device="cuda").manual_seed(4)
    g = torch.view_as_complex(torch.randn((4096, 2 * ng, 2), dtype=torch.float64, device="cuda", generator=gen))
    chi = K.bubble_irrq(g.reshape(nk + (1, 1, 2 * ng)), nk, niw, niv, beta, K.to_dev(np.zeros(1), torch.int32))
    torch.cuda.synchronize()
    prod = (-beta / 4096) * (g.T.contiguous() @ g)  # q = 0: -beta / N sum_k G(k, v) G(k, v - w)
    for w in (0, 1, 1023, niw):
        ref = torch.diagonal(prod, -w)[ng - niv - w:ng + niv - w]  # elements (v, v - w)
        assert float((chi[w, 0, :, 0] - ref).abs().max()) < 1e-12 * float(prod.abs().max()), w
