"""J and K at the sizes where the sums over partial tiles change their shape, on an MI355X.

The reductions pick their strip height from the number of output tiles and
split the partial slots over thread groups, so the sizes cover one tile with
many slots, tile edges and remainders, and every strip height.
"""

from __future__ import annotations

import numpy as np
import pytest

from hafnium_amd import synthetic

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 1), (2, 700, 1), (100, 1200, 20), (127, 40, 5), (128, 9, 64), (129, 300, 33), (257, 97, 64),
          (385, 33, 7), (640, 24, 10), (1290, 3, 2)]


def _bound(terms, magnitude):
    """Rounding bound of sums of ``terms`` products whose absolute values sum to ``magnitude``."""
    return (terms + 16) * 2.0 ** -53 * magnitude


@pytest.mark.parametrize("nao,naux,nocc", SHAPES)
def test_occupied_build_within_the_rounding_bound(nao, naux, nocc):
    from hafnium_amd.coulomb_exchange import MI355XCoulombExchange

    b = synthetic.tensor_full(3, naux, nao)
    c = synthetic.occupied_orbitals(3, nao, nocc)
    jk = MI355XCoulombExchange(b)
    j, k = jk.jk_occupied(c)
    x, xa = b @ c, np.abs(b) @ np.abs(c)
    gamma, gamma_a = np.einsum("qmi,mi->q", x, c), np.einsum("qmi,mi->q", xa, np.abs(c))
    j_abs = np.einsum("q,qmn->mn", gamma_a, np.abs(b))
    k_abs = np.tensordot(xa, xa, axes=((0, 2), (0, 2)))
    # The reference sums round too: twice the bound.
    assert np.all(np.abs(j - np.einsum("q,qmn->mn", gamma, b)) <= 2 * _bound(naux + nao * (nocc + 1), j_abs))
    assert np.all(np.abs(k - np.tensordot(x, x, axes=((0, 2), (0, 2)))) <= 2 * _bound(naux * nocc + 2 * nao, k_abs))
    np.testing.assert_array_equal(k, k.T)
    np.testing.assert_array_equal(j, j.T)
    j2, k2 = jk.jk_occupied(c)
    np.testing.assert_array_equal(j, j2)
    np.testing.assert_array_equal(k, k2)
    np.testing.assert_allclose(jk.coulomb(c @ c.T), j, rtol=0, atol=4 * np.max(_bound(naux + nao * (nocc + 1), j_abs)))


@pytest.mark.parametrize("nao,naux", [(1, 3), (33, 40), (129, 12), (300, 5)])
def test_non_symmetric_density(nao, naux):
    """The symmetric-plus-antisymmetric reduction, diagonal tiles included."""
    from hafnium_amd.coulomb_exchange import MI355XCoulombExchange

    b = synthetic.tensor_full(5, naux, nao)
    d = synthetic.tensor_full(6, 2, nao)[0] + np.triu(synthetic.tensor_full(7, 1, nao)[0], 1)
    k = MI355XCoulombExchange(b).exchange(d)
    expect = np.einsum("qmn,nl,qls->ms", b, d, b, optimize=True)
    # Products of the eigenvectors of D: its norm and the eigensolver's rounding (n eps) scale the error.
    top = np.einsum("qmn->", np.abs(b).max(axis=(1, 2), keepdims=True) ** 2) * nao * np.linalg.norm(d, 2)
    assert np.max(np.abs(k - expect)) <= 64 * nao * 2.0 ** -53 * top


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x3"])
def test_batch_equals_single_builds(precision):
    import torch

    from hafnium_amd.batch import BatchedCoulombExchange
    from hafnium_amd.coulomb_exchange import MI355XCoulombExchange
    from tests.tolerances import BF16X3_REL_TOL, FP32_REL_TOL

    shapes = [(1, 2, 1), (31, 300, 31), (64, 7, 3), (127, 50, 40), (129, 50, 33), (260, 11, 70)]
    batch = BatchedCoulombExchange(shapes)
    tensors = [synthetic.tensor_full(i, q, n) for i, (n, q, _) in enumerate(shapes)]
    orbitals = [synthetic.occupied_orbitals(i, n, o) for i, (n, _, o) in enumerate(shapes)]
    batch.set_tensors(tensors)
    packed = batch.pack_orbitals(orbitals)
    j1, k1 = batch.run(packed, precision=precision)
    j2, k2 = batch.run(packed, batch.pack_matrices([c @ c.T for c in orbitals]), precision=precision)
    torch.cuda.synchronize()
    tol = {"fp64": 1e-12, "fp32": FP32_REL_TOL, "bf16x3": BF16X3_REL_TOL}[precision]  # fp64: 2e4 products, 2e4 2^-53
    for i, (b, c) in enumerate(zip(tensors, orbitals)):
        j, k = MI355XCoulombExchange(b).jk_occupied(c)
        for got, want in ((j1, j), (j2, j), (k1, k), (k2, k)):
            m = batch.matrix(got, i).cpu().numpy()
            assert np.max(np.abs(m - want)) <= tol * np.max(np.abs(want)), (precision, i)
            np.testing.assert_array_equal(m, m.T)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("nao,nocc", [(1, 1), (16, 16), (17, 17), (31, 5), (33, 33), (145, 129), (145, 144), (205, 145),
                                      (420, 390)])
def test_half_transform_column_groups(precision, nao, nocc):
    """Every split of the columns into groups (one, several, a narrower last one) and both workgroup sizes."""
    from hafnium_amd import _lib
    from hafnium_amd.coulomb_exchange import MI355XCoulombExchange
    from tests.tolerances import FP32_REL_TOL

    naux = 5
    b = synthetic.tensor_full(8, naux, nao)
    c = synthetic.occupied_orbitals(8, nao, nocc)
    x, xa = b @ c, np.abs(b) @ np.abs(c)
    expect = np.tensordot(x, x, axes=((0, 2), (0, 2)))
    bound = 2 * _bound(naux * nocc + 2 * nao, np.tensordot(xa, xa, axes=((0, 2), (0, 2))))
    jk = MI355XCoulombExchange(b, precision=precision)
    first = None
    for columns in (0, 32, 64, 128, 256):
        for rows in (64, 128):
            jk.set_tuning(_lib.TUNE_X_BN, columns)
            jk.set_tuning(_lib.TUNE_X_BM, rows)
            j, k = jk.jk_occupied(c)
            if precision == "fp64":
                assert np.all(np.abs(k - expect) <= bound)
            else:
                assert np.max(np.abs(k - expect)) <= FP32_REL_TOL * np.max(np.abs(expect))
            # The grouping changes neither the products nor their order.
            first = (j, k) if first is None else first
            np.testing.assert_array_equal(k, first[1])
            np.testing.assert_array_equal(j, first[0])


@pytest.mark.parametrize("length", [0, 1, 63, 1024, 8191, 8192, 8193, 70001])
def test_batched_dots(length):
    """1024 threads with eight pairs each: both sides of one round of loads, a remainder, nothing."""
    import torch

    from hafnium_amd import _lib
    from hafnium_amd.coulomb_exchange import _Context, _ptr, _stream

    count, slots = 3, 4
    g = torch.Generator(device="cuda:0").manual_seed(length)
    hist = torch.randn((slots, count, max(length, 1)), generator=g, dtype=torch.float64, device="cuda:0")
    stream = _stream(torch, hist.device)
    context = _Context(0)
    lib = _lib.load()
    out = torch.full((count,), 7.0, dtype=torch.float64, device="cuda:0")
    stride = max(length, 1)
    _lib.check(lib.hfjk_ddot_batched(context.handle, count, length, _ptr(hist[0]), stride, _ptr(hist[1]), stride,
                                     _ptr(out), stream))
    dots = torch.full((count, slots), 7.0, dtype=torch.float64, device="cuda:0")
    if length:
        _lib.check(lib.hfjk_history_dots_batched(context.handle, count, length, slots, _ptr(hist), 2, _ptr(dots),
                                                 stream))
    torch.cuda.synchronize()
    h = hist[:, :, :length].cpu().numpy().astype(np.longdouble)
    # A sum of n products in any order: n eps sum |x y|.
    for i in range(count):
        bound = max(length, 1) * 2.3e-16 * float(np.abs(h[0, i] * h[1, i]).sum())
        assert abs(float(out[i]) - float((h[0, i] * h[1, i]).sum())) <= bound
        for a in range(slots if length else 0):
            bound = length * 2.3e-16 * float(np.abs(h[2, i] * h[a, i]).sum())
            assert abs(float(dots[i, a]) - float((h[2, i] * h[a, i]).sum())) <= bound


@pytest.mark.parametrize("nao,rank", [(1, 1), (2, 2), (63, 1), (64, 63), (65, 64), (192, 65), (193, 128), (512, 130),
                                      (513, 40), (700, 200), (1025, 150)])
def test_density_factor_in_panels_and_in_steps(nao, rank):
    """Every number of thread groups, panels that end at, before and after the rank, and the change to steps."""
    from hafnium_amd.coulomb_exchange import MI355XCoulombExchange

    naux = 3
    b = synthetic.tensor_full(5, naux, nao)
    rng = np.random.default_rng(nao + rank)
    c = rng.standard_normal((nao, rank)) * np.geomspace(1.0, 0.1, rank)
    d = c @ c.T
    jk = MI355XCoulombExchange(b)
    k = jk.exchange(d)
    x = b @ c
    expect = np.tensordot(x, x, axes=((0, 2), (0, 2)))
    # The factor's residual, checked by the library, is at most 1e-11 max |D|, and
    # each element of D enters K through products of two rows of B.
    rows = np.abs(b).sum(axis=2)
    assert np.all(np.abs(k - expect) <= 2e-11 * np.abs(d).max() * np.einsum("qm,qn->mn", rows, rows))
    np.testing.assert_array_equal(k, k.T)


@pytest.mark.parametrize("precision", ["fp32", "bf16x3"])
@pytest.mark.parametrize("nao,naux,nocc", [(9, 1, 1), (24, 84, 5), (96, 336, 20), (130, 257, 33), (192, 512, 64),
                                           (192, 672, 40), (300, 700, 130)])
def test_short_runs_of_the_single_precision_syrk(precision, nao, naux, nocc):
    """Runs from four aux functions to 4096 products, one workgroup per run or several runs, both stream orders."""
    from hafnium_amd import _lib
    from hafnium_amd.coulomb_exchange import MI355XCoulombExchange
    from tests.tolerances import BF16X3_REL_TOL, FP32_REL_TOL

    b = synthetic.tensor_full(11, naux, nao)
    c = synthetic.occupied_orbitals(11, nao, nocc)
    x = b @ c
    k_ref = np.tensordot(x, x, axes=((0, 2), (0, 2)))
    j_ref = np.tensordot(np.einsum("qmi,mi->q", x, c), b, axes=(0, 0))
    tol = FP32_REL_TOL if precision == "fp32" else BF16X3_REL_TOL
    jk = MI355XCoulombExchange(b, precision=precision)
    for splits, serial in ((0, 0), (0, 1), (8, 0), (200, 0)):
        jk.set_tuning(_lib.TUNE_SYRK_SPLITS, splits)
        jk.set_tuning(_lib.TUNE_COULOMB_SERIAL, serial)
        j, k = jk.jk_occupied(c)
        assert np.max(np.abs(k - k_ref)) <= tol * np.max(np.abs(k_ref))
        assert np.max(np.abs(j - j_ref)) <= tol * np.max(np.abs(j_ref))


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x3"])
@pytest.mark.parametrize("nao,naux,nocc", [(9, 1, 1), (24, 84, 5), (96, 336, 20), (130, 257, 33), (192, 672, 40),
                                           (260, 640, 250), (260, 700, 250)])
def test_runs_of_signed_columns(precision, nao, naux, nocc):
    """Signed columns: runs of a round, of two rounds (the last shape) and at the limit of products, split counts of
    their own and given ones."""
    from hafnium_amd import _lib
    from hafnium_amd.coulomb_exchange import MI355XCoulombExchange
    from tests.tolerances import BF16X3_REL_TOL, FP32_REL_TOL, FP64_REL_TOL

    b = synthetic.tensor_full(13, naux, nao)
    c = synthetic.occupied_orbitals(13, nao, nocc)
    signs = np.where(np.arange(nocc) % 3 == 1, -1.0, 1.0)
    x = b @ c
    k_ref = np.tensordot(x * signs, x, axes=((0, 2), (0, 2)))
    scale = np.max(np.abs(np.tensordot(x, x, axes=((0, 2), (0, 2)))))  # the sum of magnitudes' size
    tol = {"fp64": FP64_REL_TOL, "fp32": FP32_REL_TOL, "bf16x3": BF16X3_REL_TOL}[precision]
    jk = MI355XCoulombExchange(b, precision=precision)
    for splits in (0, 8, 200):
        jk.set_tuning(_lib.TUNE_SYRK_SPLITS, splits)
        assert np.max(np.abs(jk.exchange_occupied(c, signs) - k_ref)) <= tol * scale, splits
