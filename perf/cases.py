"""The workloads whose speed is watched: what a program using this package calls, over the sizes it meets.

Each case is a dict of plain values with a ``kind``:

* ``jk``: ``MI355XCoulombExchange`` on one molecule's fitted tensor. ``entry`` "occupied" is J and K of
  D = C C^T in one call (the Fock build of the SCF), "density" the two protocol calls ``coulomb(D)`` and
  ``exchange(D)`` of a program that holds a density only.
* ``batch``: ``BatchedCoulombExchange`` on many uneven molecules (nao ~ U{40..400}).
* ``kpoint``: J and K of ``KPointMI355XCoulombExchange`` over a k-point mesh.
* ``integrals``: the metric and three-centre integrals of a water cluster on the GPU.
* ``scf_step``: one iteration of the batched SCF of water clusters (diagonalisation and density, Fock
  build, orbital gradient).
* ``mlp``: one training step of the learned guess's network.

``prepare`` makes the inputs from the seed and the objects a program keeps, ``run`` is one pass,
``exact`` the same results from plain torch in 64 bits.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

from hafnium_amd.batch import BatchedCoulombExchange
from hafnium_amd.batch_scf import BatchedRhf, atomic_start, molecule_inputs
from hafnium_amd.clusters import AUX_BASIS, ORBITAL_BASIS, atomic_density_guess
from hafnium_amd.coulomb_exchange import MI355XCoulombExchange
from hafnium_amd.integrals import metric_device, three_center_device
from hafnium_amd.kpoint import KPointMI355XCoulombExchange
from hafnium_amd.mlp import Mlp
from hafnium_amd.molecule import BasisOnAtoms, load_basis, water_cluster

DEVICE = "cuda:0"
DECAY = 20.0  # range of the fitted tensor's envelope, as in the package's synthetic workloads


def listed():
    return [
        # The benchmark's small configuration: one Fock build of a few waters, where launches and latency count.
        {"name": "jk_small_fp64", "kind": "jk", "entry": "occupied", "precision": "fp64", "full": False,
         "nao": 100, "naux": 300, "nocc": 20},
        # Fock build of twelve waters in cc-pVDZ / def2-universal-jkfit, the package's own SCF workload.
        {"name": "jk_cluster_fp64", "kind": "jk", "entry": "occupied", "precision": "fp64", "full": False,
         "nao": 288, "naux": 1356, "nocc": 60},
        # Reduced-precision build at ragged sizes (the early iterations of a mixed SCF).
        {"name": "jk_ragged_fp32", "kind": "jk", "entry": "occupied", "precision": "fp32", "full": False,
         "nao": 709, "naux": 2503, "nocc": 117},
        # A program that holds a density and no orbitals: the reference protocol's two calls.
        {"name": "jk_density_fp64", "kind": "jk", "entry": "density", "precision": "fp64", "full": False,
         "nao": 501, "naux": 1800, "nocc": 90},
        # The benchmark's large basis (nao 1500, nocc 250) with the full copy of B, on 2000 aux functions.
        {"name": "jk_large_fp64", "kind": "jk", "entry": "occupied", "precision": "fp64", "full": True,
         "nao": 1500, "naux": 2000, "nocc": 250},
        {"name": "jk_large_bf16x3", "kind": "jk", "entry": "occupied", "precision": "bf16x3", "full": True,
         "nao": 1500, "naux": 2000, "nocc": 250},
        # A quarter of the benchmark's batch of 512 uneven instances; with densities as it passes them, and
        # from the orbitals alone as the batched SCF does.
        {"name": "batch_fp64", "kind": "batch", "precision": "fp64", "densities": True, "count": 128,
         "lo": 40, "hi": 400},
        {"name": "batch_bf16x3", "kind": "batch", "precision": "bf16x3", "densities": False, "count": 128,
         "lo": 40, "hi": 400},
        # A primitive cell of two first-row atoms in a double-zeta basis on a 2 x 2 x 2 mesh.
        {"name": "kpoint", "kind": "kpoint", "nkpt": 8, "nao": 28, "naux": 212, "nocc": 4},
        # Inputs of one SCF: the integrals of twelve waters.
        {"name": "integrals", "kind": "integrals", "basis": "cc-pvdz", "waters": 12},
        # One iteration of a batch of clusters of 2 .. 12 waters.
        {"name": "scf_step", "kind": "scf_step", "count": 12, "small": 2, "large": 12},
        # The learned guess's network for oxygen, one minibatch of 256 atoms.
        {"name": "mlp_train", "kind": "mlp", "rows": 256, "hidden": 256, "outputs": 77},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["jk", "jk", "jk", "jk", "batch", "batch", "kpoint", "integrals", "scf_step", "mlp"])
    if kind == "jk":
        nao = _log_int(rng, 24, 1500)
        naux = max(8, int(nao * rng.uniform(2.5, 5.0)))
        naux = min(naux, int(4.5e9 / nao ** 2))
        nocc = max(1, int(nao * rng.uniform(0.05, 0.3)))
        nocc = max(1, min(nocc, int(3.3e12 / (3.0 * naux * nao ** 2))))
        precision = rng.choice(["fp64", "fp64", "fp32", "bf16x3"])
        return {"kind": "jk", "entry": rng.choice(["occupied", "occupied", "density"]), "precision": precision,
                "full": rng.random() < 0.3, "nao": nao, "naux": naux, "nocc": nocc}
    if kind == "batch":
        lo = rng.randint(16, 120)
        hi = rng.randint(lo + 1, 400)
        count = max(2, min(_log_int(rng, 4, 200), int(128 * (220.0 / hi) ** 3)))
        return {"kind": "batch", "precision": rng.choice(["fp64", "fp64", "bf16x3", "fp32"]),
                "densities": rng.random() < 0.5, "count": count, "lo": lo, "hi": hi}
    if kind == "kpoint":
        nkpt = rng.choice([1, 2, 3, 4, 6, 8, 12])
        nao = rng.randint(8, 64 if nkpt > 4 else 120)
        return {"kind": "kpoint", "nkpt": nkpt, "nao": nao, "naux": int(nao * rng.uniform(3.0, 8.0)),
                "nocc": max(1, int(nao * rng.uniform(0.08, 0.3)))}
    if kind == "integrals":
        return {"kind": "integrals", "basis": rng.choice(["cc-pvdz", "cc-pvdz", "def2-svp", "sto-3g"]),
                "waters": rng.randint(1, 14)}
    if kind == "scf_step":
        small = rng.randint(1, 6)
        return {"kind": "scf_step", "count": rng.randint(2, 16), "small": small, "large": rng.randint(small, 12)}
    return {"kind": "mlp", "rows": _log_int(rng, 24, 2048), "hidden": rng.choice([96, 128, 200, 256, 384]),
            "outputs": rng.randint(18, 110)}


# ------------------------------------------------------------------ inputs

def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _tensor(g, naux, nao):
    """Symmetric ``[naux, nao, nao]`` with normal entries under an exponential envelope in |m - n|."""
    at = torch.arange(nao, device=DEVICE, dtype=torch.float64)
    envelope = torch.exp(-(at[:, None] - at[None, :]).abs() / DECAY) / math.sqrt(2.0)
    out = torch.empty((naux, nao, nao), dtype=torch.float64, device=DEVICE)
    step = max(1, int(2.5e8) // (nao * nao))
    for q in range(0, naux, step):
        z = torch.randn((min(step, naux - q), nao, nao), generator=g, dtype=torch.float64, device=DEVICE)
        torch.add(z, z.transpose(1, 2), out=out[q:q + step])
        out[q:q + step] *= envelope
    return out


def _orbitals(g, nao, nocc):
    """Orthonormal ``[nao, nocc]`` columns."""
    z = torch.randn((nao, nocc), generator=g, dtype=torch.float64, device=DEVICE)
    return torch.linalg.qr(z)[0].contiguous()


def _jk_inputs(case, seed):
    g = _generator(seed)
    c = _orbitals(g, case["nao"], case["nocc"])
    return c, _tensor(g, case["naux"], case["nao"])


def _batch_shapes(case, seed):
    """Uneven instances; the sizes belong to the case, not to the seed."""
    del seed
    rng = random.Random(1000 + 7 * case["count"] + case["lo"] + case["hi"])
    shapes = []
    for _ in range(case["count"]):
        nao = rng.randint(case["lo"], case["hi"])
        shapes.append((nao, int(round(3.5 * nao)), max(1, int(round(rng.uniform(0.1, 0.3) * nao)))))
    return shapes


def _kpoint_inputs(case, seed):
    g = _generator(seed)
    nk, nao, naux, nocc = case["nkpt"], case["nao"], case["naux"], case["nocc"]
    c64 = torch.complex128
    b = torch.randn((nk, nk, naux, nao, nao), generator=g, dtype=c64, device=DEVICE)
    # The blocks of transfer zero are Hermitian, as the real pair densities of a crystal are.
    for k in range(nk):
        b[k, k] = 0.5 * (b[k, k] + b[k, k].conj().transpose(1, 2))
    sig = torch.ones((nk, nk, naux), dtype=torch.float64, device=DEVICE)
    sig[:, :, naux - naux // 16:] = -1.0  # the few negative directions of a two-dimensional or truncated metric
    w = torch.full((nk,), 1.0 / nk, dtype=torch.float64, device=DEVICE)
    a = torch.randn((nk, nao, nao), generator=g, dtype=c64, device=DEVICE) / (4.0 * nao)
    s = torch.eye(nao, dtype=c64, device=DEVICE) + a + a.conj().transpose(1, 2)
    orb = torch.linalg.qr(torch.randn((nk, nao, nocc), generator=g, dtype=c64, device=DEVICE))[0].contiguous()
    d = torch.matmul(orb, orb.conj().transpose(1, 2).contiguous())
    d = 0.5 * (d + d.conj().transpose(1, 2)).contiguous()
    return b, sig, w, s, 0.7, d


def _clusters(case, seed):
    sizes = np.linspace(case["small"], case["large"], case["count"])
    return [water_cluster(int(round(k)), 1000 * int(seed) + i) for i, k in enumerate(sizes)]


_ATOMS: dict = {}  # the spherical atoms' densities, the same for every cluster


def prepare(case, seed):
    kind = case["kind"]
    if kind == "jk":
        c, b = _jk_inputs(case, seed)
        jk = MI355XCoulombExchange(b, precision=case["precision"])
        del b
        if case["full"]:
            jk.expand_full(case["precision"])
        jk.packed_tensor(case["precision"])
        return {"kind": kind, "entry": case["entry"], "jk": jk,
                "x": c if case["entry"] == "occupied" else torch.matmul(c, c.T.contiguous())}
    if kind == "batch":
        g = _generator(seed)
        shapes = _batch_shapes(case, seed)
        batch = BatchedCoulombExchange(shapes)
        orbitals = [_orbitals(g, n, o) for n, _, o in shapes]
        for i, (n, q, _) in enumerate(shapes):
            batch.set_tensor(i, _tensor(g, q, n))
        c = batch.pack_orbitals(orbitals)
        d = batch.pack_matrices([torch.matmul(x, x.T.contiguous()) for x in orbitals]) if case["densities"] else None
        return {"kind": kind, "batch": batch, "c": c, "d": d, "precision": case["precision"]}
    if kind == "kpoint":
        b, sig, w, s, madelung, d = _kpoint_inputs(case, seed)
        return {"kind": kind, "jk": KPointMI355XCoulombExchange(b, sig, w, s, madelung), "d": d}
    if kind == "integrals":
        molecule = water_cluster(case["waters"], seed)
        return {"kind": kind, "orbital": BasisOnAtoms(case["basis"], molecule), "aux": BasisOnAtoms(AUX_BASIS, molecule)}
    if kind == "scf_step":
        molecules = _clusters(case, seed)
        for m in molecules[:1]:
            atomic_density_guess(m, cache=_ATOMS)
        batch = BatchedRhf([molecule_inputs(m) for m in molecules])
        return {"kind": kind, "batch": batch, "fock": atomic_start(batch, _ATOMS).fock}
    g = _generator(seed)
    net = Mlp([288, case["hidden"], case["hidden"], case["outputs"]], seed=seed)
    n = 4 * case["rows"]
    return {"kind": kind, "net": net,
            "x": torch.randn((n, 288), generator=g, dtype=torch.float32, device=DEVICE),
            "y": torch.randn((n, case["outputs"]), generator=g, dtype=torch.float32, device=DEVICE),
            "rows": (torch.randperm(n, generator=g, device=DEVICE).to(torch.int32), case["rows"], 2 * case["rows"])}


# ------------------------------------------------------------------ one pass

def run(state):
    kind = state["kind"]
    if kind == "jk":
        jk, x = state["jk"], state["x"]
        if state["entry"] == "occupied":
            j, k = jk.jk_occupied(x)
        else:
            j, k = jk.coulomb(x), jk.exchange(x)
        return {"J": j, "K": k}
    if kind == "batch":
        j, k = state["batch"].run(state["c"], state["d"], precision=state["precision"])
        return {"J": j, "K": k}
    if kind == "kpoint":
        return {"J": state["jk"].coulomb(state["d"]), "K": state["jk"].exchange(state["d"])}
    if kind == "integrals":
        return {"metric": metric_device(state["aux"]), "three_center": three_center_device(state["aux"], state["orbital"])}
    if kind == "scf_step":
        batch = state["batch"]
        density, _, orbitals = batch.solve(state["fock"])
        fock, gradient = torch.empty_like(density), torch.empty_like(density)
        terms = torch.empty((3, batch.count), dtype=torch.float64, device=density.device)
        batch.fock(density, orbitals, "fp64", fock, terms)
        batch.gradient(fock, density, gradient)
        return {"density": density, "fock": fock, "gradient": gradient, "terms": terms}
    net = state["net"]
    loss = net.train_step(state["x"], state["y"], state["rows"], lr=1e-3, weight_decay=1e-2)
    return {"loss": loss, "grads": net.grads, "params": net.params}


# ------------------------------------------------------------------ what a pass cannot do without

def _jk_work(nao, naux, nocc, size, density=False):
    tensor = naux * nao * (nao + 1) / 2.0
    flops = 2.0 * naux * nao ** 2 * nocc + naux * nao * (nao + 1.0) * nocc + 4.0 * tensor
    vectors = 8.0 * nao * (nao if density else nocc)
    return tensor * size + vectors + 16.0 * nao ** 2, flops


def _shells(name, molecule):
    """(l, primitives, contractions) of every shell of the molecule."""
    data = load_basis(name)
    return [(s["l"], len(s["exponents"]), len(s["coefficients"])) for z in molecule.charges for s in data[str(z)]]


def _functions(shells):
    return sum((2 * l + 1) * c for l, _, c in shells)


def work(case):
    kind = case["kind"]
    if kind == "jk":
        b, f = _jk_work(case["nao"], case["naux"], case["nocc"], 8 if case["precision"] == "fp64" else 4,
                        case["entry"] == "density")
        return {"bytes": b, "flops": f}
    if kind == "batch":
        parts = [_jk_work(n, q, o, 8 if case["precision"] == "fp64" else 4) for n, q, o in _batch_shapes(case, 0)]
        return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}
    if kind == "kpoint":
        nk, n, q, o = case["nkpt"], case["nao"], case["naux"], case["nocc"]
        return {"bytes": 16.0 * nk * nk * q * n * n + 48.0 * nk * n * n,
                "flops": 8.0 * nk * nk * q * n * n * o + 4.0 * nk * nk * q * n * n * o + 16.0 * nk * q * n * n}
    if kind == "integrals":
        molecule = water_cluster(case["waters"], 0)
        orb, aux = _shells(case["basis"], molecule), _shells(AUX_BASIS, molecule)
        n, q = _functions(orb), _functions(aux)
        # Per primitive triple: the Hermite integrals contracted with the aux function, then with the pair.
        hermite = lambda l: (l + 1) * (l + 2) * (l + 3) // 6  # noqa: E731
        cart = lambda l: (l + 1) * (l + 2) // 2  # noqa: E731
        pairs: dict = {}
        for i, (la, pa, _) in enumerate(orb):
            for lb, pb, _ in orb[:i + 1]:
                key = (max(la, lb), min(la, lb))
                pairs[key] = pairs.get(key, 0) + pa * pb
        flops = 0.0
        for (la, lb), count in pairs.items():
            h, c = hermite(la + lb), cart(la) * cart(lb)
            for lp, pp, _ in aux:
                flops += count * pp * 2.0 * (h * hermite(lp) * cart(lp) + c * h * cart(lp)) / 2.0
        return {"bytes": 8.0 * (q * n * n + q * q), "flops": flops}
    if kind == "scf_step":
        total_b = total_f = 0.0
        for m in _clusters(case, 0):
            n, q = _functions(_shells(ORBITAL_BASIS, m)), _functions(_shells(AUX_BASIS, m))
            o = m.n_electrons // 2
            b, f = _jk_work(n, q, o, 8)
            # Transform, tridiagonal reduction, back-transform and density; then the gradient's products.
            total_f += f + 4.0 * n ** 3 + 4.0 / 3.0 * n ** 3 + 2.0 * n * n * o * 3 + 8.0 * n ** 3
            total_b += b + 8.0 * n * n * 6
        return {"bytes": total_b, "flops": total_f}
    sizes = [288, case["hidden"], case["hidden"], case["outputs"]]
    params = sum(a * b + b for a, b in zip(sizes[:-1], sizes[1:]))
    m = case["rows"]
    return {"bytes": params * 4.0 * 7 + m * (288 + case["outputs"]) * 4.0,
            "flops": 2.0 * m * (3.0 * params - sizes[0] * sizes[1])}


# ------------------------------------------------------------------ results in 64 bits

def _jk_exact(c, b):
    """J and K of D = C C^T from the full tensor, in slices of aux functions."""
    naux, nao, _ = b.shape
    d = torch.matmul(c, c.T.contiguous())
    j = torch.zeros_like(d)
    k = torch.zeros_like(d)
    step = max(1, int(2e8) // (nao * max(nao, 1)))
    for q in range(0, naux, step):
        part = b[q:q + step]
        flat = part.reshape(part.shape[0], nao * nao)
        j += torch.mv(flat.T, torch.mv(flat, d.reshape(-1))).view(nao, nao)
        x = torch.matmul(part.reshape(-1, nao), c).view(part.shape[0], nao, -1)
        x = x.transpose(0, 1).reshape(nao, -1).contiguous()
        k += torch.matmul(x, x.T.contiguous())
    return j, k


def _scf_exact(case, seed):
    state = prepare(case, seed)
    batch, fock = state["batch"], state["fock"]
    nm = batch.nm
    zeros = lambda: torch.zeros((batch.count, nm, nm), dtype=torch.float64, device=DEVICE)  # noqa: E731
    density, out, gradient = zeros(), zeros(), zeros()
    terms = torch.zeros((3, batch.count), dtype=torch.float64, device=DEVICE)
    for i, inp in enumerate(batch.inputs):
        n, kept = inp.nao, batch.kept[i].bool()
        x = batch.x[i][:n][:, kept].contiguous()
        f = torch.matmul(x.T.contiguous(), torch.matmul(fock[i, :n, :n].contiguous(), x))
        v = torch.linalg.eigh((0.5 * (f + f.T)).cpu())[1].to(DEVICE)
        c = torch.matmul(x, v[:, :inp.n_alpha].contiguous())
        factor = torch.linalg.cholesky(torch.as_tensor(inp.metric).cpu())
        three = torch.as_tensor(inp.three_center).cpu().reshape(inp.naux, n * n)
        b = torch.linalg.solve_triangular(factor, three, upper=False).to(DEVICE).view(inp.naux, n, n)
        j, k = _jk_exact(c, 0.5 * (b + b.transpose(1, 2)))
        d = torch.matmul(c, c.T.contiguous())
        h, s = batch.h[i, :n, :n].contiguous(), batch.s[i, :n, :n].contiguous()
        fnew = h + 2.0 * j - k
        fds = torch.matmul(torch.matmul(fnew, d), s)
        full_x = batch.x[i][:n].contiguous()
        gradient[i] = torch.matmul(torch.matmul(full_x.T.contiguous(), fds - fds.T), full_x)
        density[i, :n, :n], out[i, :n, :n] = d, fnew
        terms[:, i] = torch.stack([(d * h).sum(), (d * j).sum(), (d * k).sum()])
    return {"density": density, "fock": out, "gradient": gradient, "terms": terms}


def _mlp_exact(case, seed):
    state = prepare(case, seed)
    net, (rows, lo, hi) = state["net"], state["rows"]
    at = rows[lo:hi].long()
    x, y = state["x"][at].double(), state["y"][at].double()
    params = net.params.double()
    layers = [(params[w:b].view(k, n), params[b:b + n])
              for (w, b), k, n in zip(net.offsets, net.sizes[:-1], net.sizes[1:])]
    inputs, pre, h = [], [], x
    for i, (w, b) in enumerate(layers):
        inputs.append(h)
        z = torch.matmul(h, w) + b
        pre.append(z)
        h = z if i == len(layers) - 1 else z * torch.sigmoid(z)
    m = x.shape[0]
    loss = ((h - y) ** 2).sum() / m
    dz, grads = 2.0 * (h - y) / m, [None] * len(layers)
    for i in range(len(layers) - 1, -1, -1):
        grads[i] = torch.cat([torch.matmul(inputs[i].T.contiguous(), dz).reshape(-1), dz.sum(0)])
        if i:
            s = torch.sigmoid(pre[i - 1])
            dz = torch.matmul(dz, layers[i][0].T.contiguous()) * (s * (1.0 + pre[i - 1] * (1.0 - s)))
    return {"loss": loss.reshape(1), "grads": torch.cat(grads), "params": None}


def exact(case, seed):
    kind = case["kind"]
    if kind == "jk":
        j, k = _jk_exact(*_jk_inputs(case, seed))
        return {"J": j, "K": k}
    if kind == "batch":
        g = _generator(seed)
        shapes = _batch_shapes(case, seed)
        orbitals = [_orbitals(g, n, o) for n, _, o in shapes]
        parts = [_jk_exact(c, _tensor(g, q, n)) for c, (n, q, _) in zip(orbitals, shapes)]
        return {"J": torch.cat([j.reshape(-1) for j, _ in parts]), "K": torch.cat([k.reshape(-1) for _, k in parts])}
    if kind == "kpoint":
        b, sig, w, s, madelung, d = _kpoint_inputs(case, seed)
        nk, _, naux, nao, _ = b.shape
        charges = torch.zeros(naux, dtype=torch.complex128, device=DEVICE)
        for k in range(nk):
            charges += w[k] * torch.matmul(b[k, k].reshape(naux, -1).conj(), d[k].reshape(-1))
        j, x = torch.empty_like(d), torch.empty_like(d)
        for k in range(nk):
            j[k] = torch.matmul(sig[k, k] * charges, b[k, k].reshape(naux, -1)).view(nao, nao)
            acc = madelung * torch.matmul(torch.matmul(s[k], d[k]), s[k])
            for q in range(nk):
                left = torch.matmul(b[k, q].reshape(-1, nao), d[q]).view(naux, nao, nao) * sig[k, q][:, None, None]
                left = left.transpose(0, 1).reshape(nao, -1).contiguous()
                right = b[k, q].transpose(0, 1).reshape(nao, -1)
                acc = acc + w[q] * torch.matmul(left, right.conj().T.contiguous())
            x[k] = acc
        return {"J": j, "K": x}
    if kind == "scf_step":
        return _scf_exact(case, seed)
    if kind == "mlp":
        return _mlp_exact(case, seed)
    return None  # three-centre integrals: no closed form plain torch could give in the time


def tolerance(case):
    """About four times the distance of a pass from :func:`exact`, measured over the ranges."""
    kind = case["kind"]
    if kind in ("jk", "batch"):
        # FP64 up to 1e-14 (K, sums over naux nocc products); FP32 3e-7; the two bf16 parts 3.4e-6.
        return {"fp64": {"rel": 5e-14}, "fp32": {"rel": 1.2e-6}, "bf16x3": {"rel": 1.4e-5}}[case["precision"]]
    if kind == "kpoint":
        return {"rel": 5e-14}
    if kind == "integrals":
        return {"rel": 2e-13}  # the Boys function's recursion; no 64-bit result to compare with
    if kind == "scf_step":
        return {"rel": 1e-11}  # 64-bit rounding over the gap between occupied and virtual levels
    # bf16 operands: 4e-3 in the gradients; roundings that fall the other way move single updates.
    return {"rel": 1.5e-2}
