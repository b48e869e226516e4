"""k-point DF-J/K on the GPU against the k-point oracle (itself pinned by the supercell equivalence)."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import jk_ref, kpoint_ref
from tests.test_kpoint_oracle import ring

pytestmark = pytest.mark.gpu

TOL = 1e-10


def rel(a, b):
    return jk_ref.max_relative_error(np.asarray(a), np.asarray(b))


def random_hermitian(rng, nk, n, rank=None):
    a = rng.standard_normal((nk, n, n)) + 1j * rng.standard_normal((nk, n, n))
    if rank is not None:  # positive semidefinite of the given rank
        c = a[:, :, :rank]
        return c @ np.conj(np.swapaxes(c, 1, 2))
    return 0.5 * (a + np.conj(np.swapaxes(a, 1, 2)))


@pytest.mark.parametrize("ncell", [1, 3, 4])
def test_supercell_ring_matches_the_oracle(ncell):
    from hafnium_amd.kpoint import KPointMI355XCoulombExchange

    beta, d_super = ring(10 + ncell, naux=6, nao=5, ncell=ncell)
    _, b_k, _ = kpoint_ref.supercell_tensor(beta)
    d_k = kpoint_ref.from_supercell(d_super, ncell)
    sig = np.ones(b_k.shape[:3])
    sig[:, :, 1] = -1.0
    w = np.full(ncell, 1.0 / ncell)
    s = np.broadcast_to(np.eye(5), (ncell, 5, 5)).astype(np.complex128)
    jk = KPointMI355XCoulombExchange(b_k, sig, w, s, 0.0)
    assert rel(jk.coulomb(d_k), kpoint_ref.coulomb(b_k, sig, w, d_k)) < TOL
    assert rel(jk.exchange(d_k), kpoint_ref.exchange(b_k, sig, w, s, 0.0, d_k)) < TOL


@pytest.mark.parametrize("nk,naux,nao,rank", [(2, 40, 20, None), (3, 25, 33, 4), (1, 70, 64, None), (2, 9, 70, 12)])
def test_general_blocks_match_the_oracle(nk, naux, nao, rank):
    """Random complex transfer blocks, mixed signatures, uneven weights, the Madelung term, and
    indefinite or low-rank Hermitian densities."""
    from hafnium_amd.kpoint import KPointMI355XCoulombExchange

    rng = np.random.default_rng(100 * nk + nao)
    b = rng.standard_normal((nk, nk, naux, nao, nao)) + 1j * rng.standard_normal((nk, nk, naux, nao, nao))
    b *= np.exp(-np.abs(np.subtract.outer(np.arange(nao), np.arange(nao))) / 10.0)
    sig = np.where(rng.random((nk, nk, naux)) < 0.2, -1.0, 1.0)
    w = rng.random(nk) + 0.1
    w /= w.sum()
    s = random_hermitian(rng, nk, nao, rank=nao) + nao * np.eye(nao)
    d = random_hermitian(rng, nk, nao, rank=rank)
    jk = KPointMI355XCoulombExchange(b, sig, w, s, 0.29)
    assert rel(jk.coulomb(d), kpoint_ref.coulomb(b, sig, w, d)) < TOL
    assert rel(jk.exchange(d), kpoint_ref.exchange(b, sig, w, s, 0.29, d)) < TOL


def test_zero_transfer_builder_and_device_tensors():
    import torch

    from hafnium_amd.errors import InputError
    from hafnium_amd.kpoint import KPointMI355XCoulomb

    rng = np.random.default_rng(7)
    nk, naux, nao = 3, 30, 17
    b = rng.standard_normal((nk, naux, nao, nao)) + 1j * rng.standard_normal((nk, naux, nao, nao))
    sig = np.where(rng.random(naux) < 0.3, -1.0, 1.0)
    w = np.full(nk, 1.0 / nk)
    d = random_hermitian(rng, nk, nao)
    jk = KPointMI355XCoulomb(b, sig, w)
    got = jk.coulomb(torch.from_numpy(d).cuda())
    assert isinstance(got, torch.Tensor)
    assert rel(got.cpu().numpy(), kpoint_ref.coulomb_zero_transfer(b, sig, w, d)) < TOL
    with pytest.raises(InputError, match="Coulomb term alone"):
        jk.exchange(d)


def test_malformed_inputs_are_rejected():
    from hafnium_amd.errors import InputError
    from hafnium_amd.kpoint import KPointMI355XCoulombExchange

    b = np.zeros((2, 2, 3, 4, 4), dtype=complex)
    with pytest.raises(InputError, match="kpt, kpt, aux, ao, ao"):
        KPointMI355XCoulombExchange(b[0], np.ones((2, 3)), np.ones(2), np.zeros((2, 4, 4)), 0.0)
    with pytest.raises(InputError, match="signature"):
        KPointMI355XCoulombExchange(b, np.ones((2, 3)), np.ones(2), np.zeros((2, 4, 4)), 0.0)
    with pytest.raises(InputError, match="weights"):
        KPointMI355XCoulombExchange(b, np.ones((2, 2, 3)), np.ones(3), np.zeros((2, 4, 4)), 0.0)
    jk = KPointMI355XCoulombExchange(b, np.ones((2, 2, 3)), np.full(2, 0.5), np.zeros((2, 4, 4)), 0.0)
    with pytest.raises(InputError, match="not Hermitian"):
        jk.exchange(np.ones((2, 4, 4)) + 1j * np.triu(np.ones((2, 4, 4))))
    with pytest.raises(InputError, match="shape"):
        jk.coulomb(np.zeros((2, 3, 3)))


@pytest.mark.parametrize("nk,nao,naux,nocc", [(1, 2, 3, 1), (3, 4, 5, 4), (2, 17, 9, 16), (5, 31, 20, 17), (1, 130, 6, 40),
                                              (9, 12, 7, 3)])
@pytest.mark.parametrize("positive", [True, False])
def test_exchange_of_both_factorisations(nk, nao, naux, nocc, positive):
    """Positive semidefinite densities (Cholesky, whole ranges of blocks) and indefinite ones (eigenpairs, block by
    block) against the definition, with mixed signatures, uneven weights and ranks, and the Madelung term."""
    from hafnium_amd.kpoint import KPointMI355XCoulombExchange

    rng = np.random.default_rng(nk * 1000 + nao)
    z = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    b = z(nk, nk, naux, nao, nao)
    sig = np.where(rng.random((nk, nk, naux)) < 0.3, -1.0, 1.0)
    w = rng.uniform(0.2, 1.0, nk)
    s = z(nk, nao, nao)
    s = s + s.conj().transpose(0, 2, 1)
    d = np.zeros((nk, nao, nao), dtype=complex)
    for k in range(nk):
        c = z(nao, max(1, nocc - k % 3))
        d[k] = c @ c.conj().T
        if not positive and k == nk - 1:
            d[k] -= 3.0 * np.eye(nao)
        d[k] = 0.5 * (d[k] + d[k].conj().T)
    expect = np.einsum("k,qkpxy,qkp,kyz,qkpwz->qxw", w, b, sig, d, b.conj(), optimize=True)
    expect += 0.4 * s @ d @ s
    got = KPointMI355XCoulombExchange(b, sig, w, s, 0.4).exchange(d)
    # Sums of nk naux nocc products: their rounding relative to the sum of magnitudes.
    top = np.einsum("k,qkpxy,kyz,qkpwz->qxw", w, np.abs(b), np.abs(d), np.abs(b), optimize=True).max() + \
        0.4 * (np.abs(s) @ np.abs(d) @ np.abs(s)).max()
    assert np.max(np.abs(got - expect)) <= 64 * nao * 2.0 ** -53 * top
    assert np.max(np.abs(got - got.conj().transpose(0, 2, 1))) <= 16 * nao * 2.0 ** -53 * top


@pytest.mark.parametrize("nk,naux", [(4, 9000), (6, 2300)])
def test_exchange_in_several_passes(nk, naux):
    """More blocks than the workspace holds X of (1 GiB): ranges of k2 within one k1, which accumulate, and whole
    k1 a few at a time. Every block, signature and weight differs."""
    import torch

    from hafnium_amd.kpoint import KPointMI355XCoulombExchange

    nao = 40
    columns = 96  # of X for full rank: Re and Im, 40 rounded up to 16 each
    fit = (1 << 30) // (naux * nao * columns * 8)
    assert 1 < fit < nk if nk == 4 else nk <= fit < nk * nk  # ranges of k2; whole k1, not all of them
    g = torch.Generator(device="cuda:0")
    g.manual_seed(4)
    c128 = torch.complex128
    b = torch.randn((nk, nk, naux, nao, nao), generator=g, dtype=c128, device="cuda:0")
    sig = torch.where(torch.rand((nk, nk, naux), generator=g, device="cuda:0") < 0.3, -1.0, 1.0).double()
    w = torch.linspace(0.3, 1.0, nk, dtype=torch.float64, device="cuda:0")
    c = torch.randn((nk, nao, nao), generator=g, dtype=c128, device="cuda:0")
    d = torch.matmul(c, c.conj().transpose(1, 2).contiguous())
    d = 0.5 * (d + d.conj().transpose(1, 2)).contiguous()
    got = KPointMI355XCoulombExchange(b, sig, w, torch.zeros((nk, nao, nao), dtype=c128, device="cuda:0"),
                                      0.0).exchange(d)
    for k1 in range(nk):
        want = torch.zeros((nao, nao), dtype=c128, device="cuda:0")
        for k2 in range(nk):
            left = torch.matmul(b[k1, k2].reshape(-1, nao), d[k2]).view(naux, nao, nao) * sig[k1, k2][:, None, None]
            left = left.transpose(0, 1).reshape(nao, -1).contiguous()
            want += w[k2] * torch.matmul(left, b[k1, k2].transpose(0, 1).reshape(nao, -1).conj().T.contiguous())
        assert float((got[k1] - want).abs().max()) <= 1e-12 * float(want.abs().max()), k1


@pytest.mark.parametrize("extra", [-8e-12, -2e-12, 2e-12, 8e-12, 3e-11])
@pytest.mark.parametrize("spread", [False, True])
def test_exchange_keeps_small_eigenvalues_above_the_cut(extra, spread):
    """Four unit eigenvalues and a small one of either sign above 1e-12 of them, on one function or spread over
    all: it enters K in full, where the factor of a nearly semidefinite density would have dropped it."""
    from hafnium_amd.kpoint import KPointMI355XCoulombExchange

    rng = np.random.default_rng(11)
    nk, naux, nao = 2, 40, 28
    z = lambda *s: rng.standard_normal(s) + 1j * rng.standard_normal(s)  # noqa: E731
    b = z(nk, nk, naux, nao, nao)
    # The small eigenvector's products are 1e6 times the others', so that its part of K shows.
    b[..., 0] *= 1e6
    d = np.zeros((nk, nao, nao), dtype=complex)
    for k in range(nk):
        u = np.zeros((nao, 5), dtype=complex)
        u[1:, :4] = np.linalg.qr(z(nao - 1, 4))[0]
        if spread:
            u[1:, 4] = np.linalg.qr(np.concatenate([u[1:, :4], z(nao - 1, 1)], 1))[0][:, 4]
            u[:, 4] = (u[:, 4] + np.eye(nao)[0]) / np.sqrt(2.0)
        else:
            u[0, 4] = 1.0
        d[k] = (u * np.array([1.0, 1.0, 1.0, 1.0, extra])) @ u.conj().T
        d[k] = 0.5 * (d[k] + d[k].conj().T)
    w = np.full(nk, 1.0 / nk)
    got = KPointMI355XCoulombExchange(b, np.ones((nk, nk, naux)), w, np.zeros((nk, nao, nao)), 0.0).exchange(d)
    want = np.einsum("k,qkpxy,kyz,qkpwz->qxw", w, b, d, b.conj(), optimize=True)
    # D's own rounding reaches K 1e12-fold through the scaled function (1e-4 and less, from NumPy's eigenpairs);
    # without the extra eigenvalue K would be off by 0.22 and more.
    assert np.linalg.norm(got - want) <= 1e-3 * np.linalg.norm(want)
