"""MLP kernels on the GPU against the CPU oracle: GEMM forms, forward, gradients, Adam, training."""

from __future__ import annotations

import numpy as np
import pytest

from oracle import mlp_ref

pytestmark = pytest.mark.gpu

# GEMM: identical bf16 operands, FP32 (kernel) vs FP64 (oracle) sums of <= 300 terms.
GEMM_REL_TOL = 1e-5
# Whole network: intermediates rounded to bf16 can land on the other side of a
# rounding boundary when the FP32 and FP64 sums differ in the last bit, so a few
# operands differ by one bf16 ulp (2^-8 relative).
NET_REL_TOL = 2e-3


def _torch():
    import torch

    return torch


def _gemm(lib_mlp, a, b, ta, tb, rows=None, bias=None, silu=False, a16=False, b16=False):
    torch = _torch()
    dev = lib_mlp.device
    m = a.shape[1] if ta else (len(rows) if rows is not None else a.shape[0])
    k = a.shape[0] if ta else a.shape[1]
    if ta and rows is not None:
        k = len(rows)
    n = b.shape[0] if tb else b.shape[1]
    ad = torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dev)
    bd = torch.from_numpy(np.ascontiguousarray(b, dtype=np.float32)).to(dev)
    if a16:
        ad = ad.to(torch.bfloat16)
    if b16:
        bd = bd.to(torch.bfloat16)
    c = torch.empty((m, n), dtype=torch.float32, device=dev)
    h = torch.empty_like(c) if silu else None
    rows_d = None if rows is None else (torch.tensor(rows, dtype=torch.int32, device=dev), 0)
    bias_d = None if bias is None else (torch.from_numpy(bias.astype(np.float32)).to(dev), 0)
    lib_mlp._gemm(m, n, k, ad, 0, a16, a.shape[1], ta, rows_d, bd, 0, b16, b.shape[1], tb, bias_d, c, h)
    torch.cuda.synchronize()
    return c.cpu().numpy().astype(np.float64), None if h is None else h.cpu().numpy().astype(np.float64)


@pytest.fixture(scope="module")
def net():
    from hafnium_amd.mlp import Mlp

    return Mlp([72, 96, 80, 13], seed=1)


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_gemm_transpositions(net, ta, tb):
    rng = np.random.default_rng(10 + 2 * ta + tb)
    m, n, k = 131, 77, 300  # no dimension a multiple of the 64 x 64 x 32 tiles
    a = rng.standard_normal((k, m) if ta else (m, k))
    b = rng.standard_normal((n, k) if tb else (k, n))
    c, _ = _gemm(net, a, b, ta, tb)
    op_a = mlp_ref.bf16_round(a.T if ta else a)
    op_b = mlp_ref.bf16_round(b.T if tb else b)
    ref = op_a @ op_b
    assert np.abs(c - ref).max() <= GEMM_REL_TOL * np.abs(ref).max()


def test_gemm_gather_bias_silu_and_bf16_operands(net):
    rng = np.random.default_rng(20)
    x = rng.standard_normal((50, 40))
    w = rng.standard_normal((40, 70))
    bias = rng.standard_normal(70)
    rows = [49, 0, 7, 7, 31, 2, 18, 44, 5]
    c, h = _gemm(net, x, w, False, False, rows=rows, bias=bias, silu=True, b16=True)
    ref = mlp_ref.bf16_round(x[rows]) @ mlp_ref.bf16_round(w) + bias.astype(np.float32)  # bias stays FP32
    assert np.abs(c - ref).max() <= GEMM_REL_TOL * np.abs(ref).max()
    np.testing.assert_allclose(h, mlp_ref.silu(c), rtol=1e-5, atol=1e-6)
    # Transposed gathered operand: op(A) = x[rows]^T, the weight-gradient form.
    g = rng.standard_normal((len(rows), 70))
    c2, _ = _gemm(net, x, g, True, False, rows=rows)
    ref2 = mlp_ref.bf16_round(x[rows]).T @ mlp_ref.bf16_round(g)
    assert np.abs(c2 - ref2).max() <= GEMM_REL_TOL * np.abs(ref2).max()
    # bf16 storage of A gives the same result as rounding it on load.
    c3, _ = _gemm(net, x, w, False, False, a16=True)
    c4, _ = _gemm(net, x, w, False, False)
    assert np.abs(c3 - c4).max() <= GEMM_REL_TOL * np.abs(c4).max()


def test_forward_and_gradients_match_the_oracle(net):
    torch = _torch()
    rng = np.random.default_rng(30)
    x = rng.standard_normal((200, 72)).astype(np.float32)
    t = rng.standard_normal((200, 13)).astype(np.float32)
    wts = rng.uniform(0.5, 2.0, 13).astype(np.float32)
    layers = net.layers()
    xd = torch.from_numpy(x).to(net.device)
    td = torch.from_numpy(t).to(net.device)
    wd = torch.from_numpy(wts).to(net.device)
    rows = np.arange(200)[::-1].copy()
    rd = torch.from_numpy(rows.astype(np.int32)).to(net.device)
    y = net.forward(xd, (rd, 0, 200), keep=True)
    grad = torch.empty_like(y)
    loss = net.loss(y, td, (rd, 0, 200), wd, 1.0 / 200, grad)
    net.backward(grad)
    torch.cuda.synchronize()
    y_ref, _ = mlp_ref.forward(layers, x[rows], exact=False)
    assert np.abs(y.cpu().numpy() - y_ref).max() <= NET_REL_TOL * np.abs(y_ref).max()
    loss_ref, grads_ref = mlp_ref.loss_and_gradients(layers, x[rows], t[rows], wts, 1.0 / 200, exact=False)
    assert float(loss.item()) == pytest.approx(loss_ref, rel=NET_REL_TOL)
    for (dw, db), (dw_ref, db_ref) in zip(net.gradients(), grads_ref):
        assert np.abs(dw - dw_ref).max() <= NET_REL_TOL * np.abs(dw_ref).max()
        assert np.abs(db - db_ref).max() <= NET_REL_TOL * np.abs(db_ref).max()
    # And the exact (float64) network, to the size of bf16 rounding.
    _, grads_exact = mlp_ref.loss_and_gradients(layers, x[rows], t[rows], wts, 1.0 / 200, exact=True)
    for (dw, _), (dw_ex, _) in zip(net.gradients(), grads_exact):
        assert np.abs(dw - dw_ex).max() <= 5e-2 * np.abs(dw_ex).max()


def test_adam_matches_the_oracle():
    torch = _torch()
    from hafnium_amd.mlp import Mlp

    net = Mlp([8, 16, 3], seed=2)
    p0 = net.params.cpu().numpy().astype(np.float64)
    rng = np.random.default_rng(40)
    m1 = np.zeros_like(p0)
    m2 = np.zeros_like(p0)
    p = p0.copy()
    for step in range(1, 4):
        g = rng.standard_normal(p.size)
        net.grads.copy_(torch.from_numpy(g.astype(np.float32)).to(net.device))
        net.adam(1e-2, weight_decay=1e-3)
        p, m1, m2 = mlp_ref.adam_step(p, g.astype(np.float32).astype(np.float64), m1, m2, step, 1e-2,
                                      weight_decay=1e-3)
    torch.cuda.synchronize()
    np.testing.assert_allclose(net.params.cpu().numpy(), p, rtol=1e-5, atol=1e-7)
    # The bf16 copy follows the master weights.
    np.testing.assert_array_equal(net.params16.float().cpu().numpy(),
                                  mlp_ref.bf16_round(net.params.cpu().numpy()).astype(np.float32))


def test_training_fits_a_teacher_network():
    torch = _torch()
    from hafnium_amd.mlp import Mlp

    rng = np.random.default_rng(50)
    teacher = [(rng.standard_normal((16, 32)) / 4, rng.standard_normal(32) * 0.1),
               (rng.standard_normal((32, 4)) / 6, rng.standard_normal(4) * 0.1)]
    x = rng.standard_normal((2048, 16)).astype(np.float32)
    t, _ = mlp_ref.forward(teacher, x, exact=True)
    net = Mlp([16, 64, 64, 4], seed=3)
    xd = torch.from_numpy(x).to(net.device)
    td = torch.from_numpy(t.astype(np.float32)).to(net.device)
    all_rows = torch.arange(2048, dtype=torch.int32, device=net.device)
    first = float(net.loss(net.forward(xd), td).item()) / 2048
    for epoch in range(30):
        perm = torch.from_numpy(rng.permutation(2048).astype(np.int32)).to(net.device)
        for lo in range(0, 2048, 128):
            net.train_step(xd, td, (perm, lo, lo + 128), lr=3e-3)
    last = float(net.loss(net.forward(xd, (all_rows, 0, 2048)), td).item()) / 2048
    assert last < 0.05 * first


@pytest.mark.parametrize("m", [1, 33, 200])
@pytest.mark.parametrize("sizes", [[5, 3], [72, 96, 80, 13], [31, 33, 64, 65], [40, 256, 8]])
def test_training_step_is_the_separate_calls(sizes, m):
    """Tiles of 32, k split over eight waves of 32: sizes on both sides of each, operands off 16-byte lines."""
    torch = _torch()
    from hafnium_amd.mlp import Mlp

    rng = np.random.default_rng(60 + m + len(sizes))
    fused, split = Mlp(sizes, seed=4), Mlp(sizes, seed=4)
    dev = fused.device
    x = torch.from_numpy(rng.standard_normal((m + 7, sizes[0])).astype(np.float32)).to(dev)
    t = torch.from_numpy(rng.standard_normal((m + 7, sizes[-1])).astype(np.float32)).to(dev)
    w = torch.from_numpy(rng.uniform(0.5, 2.0, sizes[-1]).astype(np.float32)).to(dev)
    perm = torch.from_numpy(rng.permutation(m + 7).astype(np.int32)).to(dev)
    rows = (perm, 3, 3 + m)
    loss = fused.train_step(x, t, rows, lr=1e-2, col_weights=w, weight_decay=1e-2)
    y = split.forward(x, rows, keep=True)
    grad = torch.empty_like(y)
    loss_ref = split.loss(y, t, rows, w, 1.0 / m, grad)
    split.backward(grad)
    split.adam(1e-2, weight_decay=1e-2)
    torch.cuda.synchronize()
    # Same operands and products; the slopes multiply before the store instead of
    # after it. Only sums over at most 256 FP32 terms in another order differ.
    assert float(loss.item()) == pytest.approx(float(loss_ref.item()), rel=1e-5)
    for (dw, db), (dw_ref, db_ref) in zip(fused.gradients(), split.gradients()):
        assert np.abs(dw - dw_ref).max() <= GEMM_REL_TOL * max(np.abs(dw_ref).max(), 1e-30)
        assert np.abs(db - db_ref).max() <= GEMM_REL_TOL * max(np.abs(db_ref).max(), 1e-30)
    # A step of Adam is lr_t m1 / (sqrt(m2) + eps): its sensitivity to the gradient is checked on the moments.
    np.testing.assert_allclose(fused.moment1.cpu().numpy(), 0.1 * fused.grads.cpu().numpy(), rtol=1e-6)
    np.testing.assert_array_equal(fused.params16.float().cpu().numpy(),
                                  mlp_ref.bf16_round(fused.params.cpu().numpy()).astype(np.float32))
    # The kept activations serve a further backward pass, as the separate calls' do.
    for (h, z), (h_ref, z_ref) in zip(fused._kept()[0], split._kept()[0]):
        for got, want in ((h, h_ref), (z, z_ref)):
            assert got.shape == want.shape
            assert (got - want).abs().max().item() <= GEMM_REL_TOL * max(want.abs().max().item(), 1e-30)


@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("k", [32, 9 * 32, 16 * 32, 17 * 32 + 5, 1300])
def test_products_sum_along_k_in_order(net, k, ta, tb):
    """One product per 32 k, so the FP32 sum of an element depends on the order of the steps alone: large terms
    that swallow small ones and cancel later leave what the chain from k = 0 leaves, exactly."""
    m, n = 37, 35
    a = np.zeros((m, k))
    want = np.float32(0.0)
    for s, at in enumerate(range(0, k, 32)):
        value = (2.0 ** 30, float(s % 100 + 1), -(2.0 ** 30))[s % 3]
        a[:, at] = value
        want = np.float32(want + np.float32(value))
    c, _ = _gemm(net, a.T if ta else a, np.ones((n, k) if tb else (k, n)), ta, tb)
    np.testing.assert_array_equal(c, np.full((m, n), want, dtype=np.float64))


@pytest.mark.parametrize("m", [1, 33, 700])
@pytest.mark.parametrize("sizes", [[5, 3], [72, 96, 80, 13], [31, 33, 64, 65], [288, 256, 256, 77]])
def test_training_step_has_the_gradients_of_the_separate_calls(sizes, m):
    """The same products and sums in the same order: the same gradients and parameters, bit for bit."""
    torch = _torch()
    from hafnium_amd.mlp import Mlp

    rng = np.random.default_rng(80 + m + len(sizes))
    fused, split = Mlp(sizes, seed=6), Mlp(sizes, seed=6)
    dev = fused.device
    x = torch.from_numpy(rng.standard_normal((m + 7, sizes[0])).astype(np.float32)).to(dev)
    t = torch.from_numpy(rng.standard_normal((m + 7, sizes[-1])).astype(np.float32)).to(dev)
    rows = (torch.from_numpy(rng.permutation(m + 7).astype(np.int32)).to(dev), 3, 3 + m)
    for _ in range(2):
        fused.train_step(x, t, rows, lr=1e-3, weight_decay=1e-2)
        y = split.forward(x, rows, keep=True)
        grad = torch.empty_like(y)
        split.loss(y, t, rows, None, 1.0 / m, grad)
        split.backward(grad)
        split.adam(1e-3, weight_decay=1e-2)
        assert torch.equal(fused.grads, split.grads)
        assert torch.equal(fused.params, split.params)


def _free_memory(need):
    torch = _torch()
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < need:
        pytest.skip(f"needs {need >> 30} GiB of free GPU memory")


def test_product_of_more_tiles_than_one_grid(net):
    """8.5 million output tiles (2^32 work-items and more): an outer product of small whole numbers, exact."""
    torch = _torch()
    m, n = 4194240, 2080
    _free_memory(40 << 30)
    a = (torch.arange(m, device=net.device) % 97).float().view(m, 1)
    b = (torch.arange(n, device=net.device) % 89).float().view(1, n)
    c = torch.full((m, n), -1.0, device=net.device)
    net._gemm(m, n, 1, a, 0, False, 1, False, None, b, 0, False, n, False, None, c)
    for lo in range(0, m, m // 15):
        assert torch.equal(c[lo:lo + m // 15], a[lo:lo + m // 15] * b)


def test_training_step_of_more_tiles_than_one_grid():
    """The forward and the backward launches of 8.5 million tiles: 65535 times the same 64 rows are those rows."""
    torch = _torch()
    from hafnium_amd.mlp import Mlp

    times = 65535
    _free_memory(140 << 30)
    big, small = Mlp([1, 2080, 1], seed=9), Mlp([1, 2080, 1], seed=9)
    dev = big.device
    g = torch.Generator(device=dev)
    g.manual_seed(2)
    x = torch.randn((64, 1), generator=g, device=dev)
    t = torch.randn((64, 1), generator=g, device=dev)
    rows = torch.arange(64, dtype=torch.int32, device=dev)
    loss = big.train_step(x, t, (rows.repeat(times), 0, 64 * times), lr=1e-3)
    want = small.train_step(x, t, (rows, 0, 64), lr=1e-3)
    # Sums of 4.2 million FP32 terms in a row (the bias gradients: four chains of a million) lose up to 2^-24 of
    # the running sum each, a few 1e-3 in all; a launch's tiles left out would take half of them.
    assert float(loss.item()) == pytest.approx(float(want.item()), rel=1e-2)
    for (dw, db), (dw_ref, db_ref) in zip(big.gradients(), small.gradients()):
        assert np.linalg.norm(dw - dw_ref) <= 2e-2 * np.linalg.norm(dw_ref)
        assert np.linalg.norm(db - db_ref) <= 2e-2 * np.linalg.norm(db_ref)
    del big
    torch.cuda.empty_cache()


def test_refused_training_step_leaves_the_state():
    """A target narrower than the output is refused; the next step is then the first, as if it had not been asked."""
    torch = _torch()
    from hafnium_amd.mlp import Mlp

    net, fresh = Mlp([6, 10, 4], seed=12), Mlp([6, 10, 4], seed=12)
    g = torch.Generator(device=net.device)
    g.manual_seed(7)
    x = torch.randn((20, 6), generator=g, device=net.device)
    t = torch.randn((20, 4), generator=g, device=net.device)
    with pytest.raises(ValueError):
        net.train_step(x, t[:, :3].contiguous(), None, lr=1e-2)
    assert net.step_count == 0
    for n in (net, fresh):
        n.train_step(x, t, None, lr=1e-2)
    assert net.step_count == 1 and torch.equal(net.params, fresh.params)
