"""The GPU two- and three-centre integrals against the reference's stored PySCF values and the
(separately pinned) host engine."""

from __future__ import annotations

import time

import numpy as np
import pytest

from hafnium_amd import integrals, molecule
from tests.test_integrals import INTEGRAL_TOL

pytestmark = pytest.mark.gpu


def test_stored_metric_and_three_centre_of_water(water):
    mol = integrals.water_from_fixture_positions(water["positions_bohr"])
    orb = molecule.BasisOnAtoms("sto-3g", mol)
    aux = molecule.BasisOnAtoms("def2-universal-jkfit", mol)
    m = integrals.metric_device(aux).cpu().numpy()
    tc = integrals.three_center_device(aux, orb).cpu().numpy()
    np.testing.assert_allclose(m, water["metric"], atol=INTEGRAL_TOL * 1000, rtol=1e-12)
    np.testing.assert_allclose(tc, water["three_center"], atol=INTEGRAL_TOL * 10)


@pytest.mark.parametrize("n_waters,seed", [(1, 5), (3, 7)])
def test_device_integrals_equal_the_host_engine(n_waters, seed):
    """cc-pVDZ (general contractions, d) with def2-universal-jkfit (up to g), several centres."""
    mol = molecule.water_cluster(n_waters, seed)
    orb = molecule.BasisOnAtoms("cc-pvdz", mol)
    aux = molecule.BasisOnAtoms("def2-universal-jkfit", mol)
    m_host = integrals.metric(aux)
    tc_host = integrals.three_center(aux, orb)
    m = integrals.metric_device(aux).cpu().numpy()
    tc = integrals.three_center_device(aux, orb).cpu().numpy()
    np.testing.assert_allclose(m, m_host, atol=1e-12 * np.abs(m_host).max())
    np.testing.assert_allclose(tc, tc_host, atol=1e-12 * np.abs(tc_host).max())


def test_twelve_waters_on_the_gpu():
    """The largest cluster of the SCF workload: device against host, and the device time."""
    import torch

    mol = molecule.water_cluster(12, 112)
    orb = molecule.BasisOnAtoms("cc-pvdz", mol)
    aux = molecule.BasisOnAtoms("def2-universal-jkfit", mol)
    integrals.metric_device(aux)  # first launch: code object and tables
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    m = integrals.metric_device(aux)
    tc = integrals.three_center_device(aux, orb)
    torch.cuda.synchronize()
    seconds = time.perf_counter() - t0
    t0 = time.perf_counter()
    m_host = integrals.metric(aux)
    tc_host = integrals.three_center(aux, orb)
    host_seconds = time.perf_counter() - t0
    print(f"12 waters: device integrals {seconds:.4f} s, host {host_seconds:.4f} s", flush=True)
    np.testing.assert_allclose(m.cpu().numpy(), m_host, atol=1e-12 * np.abs(m_host).max())
    np.testing.assert_allclose(tc.cpu().numpy(), tc_host, atol=1e-12 * np.abs(tc_host).max())


class _Shells:
    """A synthetic basis in the C-ABI layout: ``(l, center, exponents, coefficient rows)`` per shell."""

    def __init__(self, shells):
        self._l = np.asarray([s[0] for s in shells], dtype=np.int32)
        self._centers = np.asarray([c for s in shells for c in s[1]], dtype=np.float64)
        self._nprim = np.asarray([len(s[2]) for s in shells], dtype=np.int32)
        self._ncontr = np.asarray([len(s[3]) for s in shells], dtype=np.int32)
        self._exps = np.asarray([e for s in shells for e in s[2]], dtype=np.float64)
        self._coefs = np.asarray([c for s in shells for row in s[3] for c in row], dtype=np.float64)
        self.n_functions = int(sum((2 * s[0] + 1) * len(s[3]) for s in shells))

    c_struct = molecule.BasisOnAtoms.c_struct


def _random_shells(rng, momenta, scale):
    out = []
    for l, nprim, ncontr in momenta:
        rows = rng.standard_normal((ncontr, nprim))
        if ncontr > 1:
            rows[0, -1] = 0.0
        out.append((l, rng.uniform(-1.5, 1.5, 3) * scale, rng.uniform(0.2, 6.0, nprim), rows))
    return out


@pytest.mark.parametrize("orbital,auxiliary", [
    # Every class of the lane-per-aux kernel, both sides of its limits, contractions on both sides.
    ([(0, 9, 3), (1, 4, 2), (2, 1, 1), (2, 3, 1)], [(0, 5, 1), (0, 1, 1), (1, 3, 2), (2, 2, 1), (3, 1, 1), (4, 1, 1), (4, 2, 1)]),
    ([(0, 1, 1), (1, 2, 1), (2, 2, 1)], [(5, 1, 1), (0, 17, 1), (1, 20, 1), (0, 16, 1), (5, 2, 1)]),
    ([(0, 2, 1), (2, 1, 1), (3, 1, 1), (3, 2, 1)], [(0, 1, 1), (1, 2, 1), (3, 1, 1)]),
    ([(0, 1, 1)], [(0, 1, 1)]),
])
@pytest.mark.parametrize("scale", [1.0, 12.0])
def test_device_integrals_over_all_classes(orbital, auxiliary, scale):
    """Both device kernels against the host engine; far centres drop primitive pairs and whole pairs."""
    rng = np.random.default_rng(7)
    orb, aux = _Shells(_random_shells(rng, orbital, scale)), _Shells(_random_shells(rng, auxiliary, scale))
    three = integrals.three_center(aux, orb)
    got = integrals.three_center_device(aux, orb).cpu().numpy()
    metric = integrals.metric(aux)
    # Each result is a sum of terms of either sign (the harmonics' Cartesian terms, the contractions) whose
    # size the Schwarz bound sqrt((P|P) (uv|uv)) gives, not the result, which far centres cancel to less;
    # (uv|uv) is below 4 for normalised functions of these exponents.
    bound = 1e-12 * np.sqrt(4.0 * np.diag(metric))[:, None, None]
    worst = float(np.max(np.abs(got - three) / bound))
    assert worst <= 1.0, worst
    np.testing.assert_array_equal(got, got.transpose(0, 2, 1))
    dev = integrals.metric_device(aux).cpu().numpy()
    worst = float(np.max(np.abs(dev - metric) / np.sqrt(np.outer(np.diag(metric), np.diag(metric)))))
    assert worst <= 1e-12, worst
    np.testing.assert_array_equal(dev, dev.T)


@pytest.mark.parametrize("momenta", [
    [(0, 5, 1), (0, 1, 1), (1, 3, 2), (2, 2, 1), (3, 1, 1), (4, 1, 1), (4, 2, 1)],
    [(0, 17, 1), (1, 16, 1), (5, 1, 1), (2, 3, 2)],
])
@pytest.mark.parametrize("shells", [224, 225])
def test_metric_of_few_and_many_shells(momenta, shells):
    """Both sides of the number of shells from which the metric goes by lanes, over all classes."""
    rng = np.random.default_rng(21)
    aux = _Shells(_random_shells(rng, [momenta[i % len(momenta)] for i in range(shells)], 4.0))
    host = integrals.metric(aux)
    dev = integrals.metric_device(aux).cpu().numpy()
    assert float(np.max(np.abs(dev - host) / np.sqrt(np.outer(np.diag(host), np.diag(host))))) <= 1e-12
    np.testing.assert_array_equal(dev, dev.T)


@pytest.mark.parametrize("distance", [13.8, 15.0, 16.5, 18.0])
def test_first_batch_of_primitive_pairs_without_a_survivor(distance):
    """Oxygens in cc-pVDZ whose first 64 of 81 s-s primitive pairs the product cut drops, and later ones not."""
    basis = molecule.load_basis("cc-pvdz")["8"]
    e = np.asarray(next(s["exponents"] for s in basis if s["l"] == 0))
    assert len(e) == 9
    kept = np.exp(-np.outer(e, e) / np.add.outer(e, e) * distance ** 2).reshape(-1) >= 1e-22
    assert not kept[:64].any() and kept[64:].any()
    positions = np.zeros((6, 3))
    positions[:, 0] = distance * np.arange(6)  # the neighbours only: the next pair has no survivor, or its own
    mol = molecule.Molecule((8,) * 6, positions)
    orb, aux = molecule.BasisOnAtoms("cc-pvdz", mol), molecule.BasisOnAtoms("def2-universal-jkfit", mol)
    host = integrals.three_center(aux, orb)
    got = integrals.three_center_device(aux, orb).cpu().numpy()
    n = orb.n_functions // 6
    for i in range(6):
        for j in range(i + 1):
            a, b = slice(i * n, (i + 1) * n), slice(j * n, (j + 1) * n)
            # Against the block's own size: the far blocks are 1e-13 of the others.
            assert np.abs(got[:, a, b] - host[:, a, b]).max() <= 1e-10 * np.abs(host[:, a, b]).max(), (i, j)


def _three_center_into(ctx, aux, orb, out, stream):
    import ctypes

    from hafnium_amd import _lib

    a, o = aux.c_struct(), orb.c_struct()
    _lib.check(ctx.lib.hfjk_int3c2e_device(ctx.handle, ctypes.byref(a), ctypes.byref(o),
                                           ctypes.c_void_p(out.data_ptr()), ctypes.c_void_p(stream.cuda_stream)))


@pytest.mark.parametrize("threads", [1, 2])
def test_integrals_beside_builds_of_the_same_context(threads):
    """The integrals and a J/K build share the context's side stream: on streams of their own, behind work that
    writes the output first, from one thread and from two, each gives what it gives alone."""
    import threading

    import torch

    from hafnium_amd import synthetic
    from hafnium_amd.coulomb_exchange import MI355XCoulombExchange

    mol = molecule.water_cluster(3, 9)
    orb, aux = molecule.BasisOnAtoms("cc-pvdz", mol), molecule.BasisOnAtoms("def2-universal-jkfit", mol)
    nao, naux, nocc = 200, 600, 30  # 7e8 products: in FP32 the Coulomb half runs on the side stream
    jk = MI355XCoulombExchange.synthetic(4, naux, nao, precision="fp32")
    c = torch.from_numpy(synthetic.occupied_orbitals(4, nao, nocc)).cuda()
    want_j, want_k = (x.clone() for x in jk.jk_occupied(c))
    want = integrals.three_center_device(aux, orb)
    load = torch.randn((2048, 2048), device="cuda:0")
    torch.cuda.synchronize()
    failures = []

    def build(times):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(times):
                j, k = jk.jk_occupied(c)
                if not (torch.equal(j, want_j) and torch.equal(k, want_k)):
                    failures.append("build")
        stream.synchronize()

    def integrate(times):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(times):
                out = torch.empty_like(want)
                for _ in range(4):
                    torch.matmul(load, load)
                out.fill_(float("nan"))  # behind the products: the integrals wait for it on every stream
                _three_center_into(jk._ctx, aux, orb, out, stream)
                if not torch.equal(out, want):
                    failures.append("integrals")
        stream.synchronize()

    if threads == 1:
        for _ in range(6):
            build(1)
            integrate(1)
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        with torch.cuda.stream(streams[0]):  # a build in flight while the integrals run
            j, k = jk.jk_occupied(c)
        out = torch.empty_like(want)
        streams[1].wait_stream(torch.cuda.current_stream())
        _three_center_into(jk._ctx, aux, orb, out, streams[1])
        torch.cuda.synchronize()
        assert torch.equal(j, want_j) and torch.equal(k, want_k) and torch.equal(out, want)
    else:
        workers = [threading.Thread(target=build, args=(20,)), threading.Thread(target=integrate, args=(20,))]
        for w in workers:
            w.start()
        for w in workers:
            w.join()
    assert not failures
