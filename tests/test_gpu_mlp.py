"""Direction-cost network: device kernels against the CPU oracle.
Tolerances: fp32 kernels 1e-4 relative (summation order differs); the bf16
MFMA inference path 3e-2 absolute on outputs of order 1 (bf16 keeps 8 bits
of mantissa)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def random_params(orc, seed, h1=32, h2=32, scale=0.5):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal(orc.mlp_nparams(h1, h2)) * scale).astype(np.float32)


def data(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.random((n, 8)).astype(np.float32)
    t = np.stack([np.sin(3 * x[:, 0]) + x[:, 1], np.cos(2 * x[:, 2]) - x[:, 3]], 1)
    return x, t.astype(np.float32)


@pytest.mark.parametrize("h1,h2", [(32, 32), (16, 8)])
def test_infer_matches_oracle(ctx, orc, h1, h2):
    p = random_params(orc, 1, h1, h2)
    x, _ = data(1000, 2)
    ctx.mlp_set(p, h1, h2)
    ref = orc.mlp_forward(p, x, h1, h2)
    np.testing.assert_allclose(ctx.mlp_infer(x, mfma=False), ref, rtol=1e-4, atol=1e-5)
    np.testing.assert_allclose(ctx.mlp_infer(x, mfma=True), ref, rtol=3e-2, atol=3e-2)


def test_grad_matches_oracle(ctx, orc):
    p = random_params(orc, 3)
    x, t = data(777, 4)
    mask = (np.random.default_rng(5).random((777, 2)) > 0.3).astype(np.float32)
    ctx.mlp_set(p)
    for mk in (None, mask):
        loss, g = ctx.mlp_loss_grad(x, t, mk)
        rloss, rg = orc.mlp_loss_grad(p, x, t, mk)
        assert loss == pytest.approx(rloss, rel=1e-4)
        np.testing.assert_allclose(g, rg, rtol=1e-3, atol=1e-5 * np.abs(rg).max())


def test_device_training_matches_oracle_adam(ctx, orc):
    p = random_params(orc, 9, scale=0.3)
    x, t = data(512, 10)
    ctx.mlp_set(p)
    loss_dev = ctx.mlp_train(x, t, epochs=20, lr=1e-2)
    q = p.copy()
    m = np.zeros_like(q)
    v = np.zeros_like(q)
    for step in range(1, 21):
        _, g = orc.mlp_loss_grad(q, x, t)
        orc.mlp_adam(q, g, m, v, 1e-2, step)
    loss_ref, _ = orc.mlp_loss_grad(q, x, t)
    got, _, _ = ctx.mlp_get()
    # Adam divides by sqrt(v): a parameter whose gradient is ~0 can move by up
    # to lr per step on either side, so compare the bulk of the parameters and
    # the loss rather than every element.
    assert np.mean(np.abs(got - q) <= 1e-3 + 1e-3 * np.abs(q)) > 0.97
    assert loss_dev == pytest.approx(loss_ref, rel=2e-2)
    first, _ = orc.mlp_loss_grad(p, x, t)
    assert loss_dev < first


@pytest.mark.parametrize("n,h1,h2", [(1, 32, 32), (31, 1, 1), (32, 32, 32), (33, 5, 17),
                                     (129, 32, 8), (8192, 32, 32), (8225, 17, 32)])
def test_grad_and_infer_at_tile_edges(ctx, orc, n, h1, h2):
    """Samples and hidden units at and beside the 32-wide tiles, the four
    waves of a workgroup and the largest grid (64 x 4 x 32 samples); the fp32
    tolerances of the tests above."""
    p = random_params(orc, 21, h1, h2)
    x, t = data(n, 22)
    mask = (np.random.default_rng(23).random((n, 2)) > 0.3).astype(np.float32)
    mask[0] = 1
    ctx.mlp_set(p, h1, h2)
    np.testing.assert_allclose(ctx.mlp_infer(x, mfma=False), orc.mlp_forward(p, x, h1, h2),
                               rtol=1e-4, atol=1e-5)
    loss, g = ctx.mlp_loss_grad(x, t, mask)
    rloss, rg = orc.mlp_loss_grad(p, x, t, mask, h1, h2)
    assert loss == pytest.approx(rloss, rel=1e-4)
    np.testing.assert_allclose(g, rg, rtol=1e-3, atol=1e-5 * np.abs(rg).max())


def test_grad_with_an_infinite_input_behind_an_idle_unit(ctx, orc):
    """An infinite activation whose successors are all idle adds nothing to
    any gradient: the result is that of any other positive input there."""
    p = random_params(orc, 31)
    p[:8] = 0
    p[0] = 1                        # unit 0 of layer 1 sees input 0 alone
    p[8:256].reshape(31, 8)[:, 0] = 0  # no other unit sees it
    p[32 * 9:32 * 9 + 1024].reshape(32, 32)[:, 0] = -50  # and it idles all of layer 2
    x, t = data(70, 32)
    x[40, 0] = 1000.0
    ctx.mlp_set(p)
    loss, g = ctx.mlp_loss_grad(x, t)
    x[40, 0] = np.inf
    for k in range(1, 32):          # 0 * inf idles the other units of that sample too
        assert p[8 * k] == 0
    loss_inf, g_inf = ctx.mlp_loss_grad(x, t)
    assert loss_inf == pytest.approx(loss, rel=1e-6)
    np.testing.assert_allclose(g_inf, g, rtol=1e-6, atol=1e-6 * np.abs(g).max())


@pytest.mark.parametrize("n", [21845, 21846, 32769])
def test_samples_on_both_sides_of_the_staged_megabyte(ctx, orc, n):
    """Samples of up to 1 MB are staged in pinned memory, more are copied; the
    fp32 tolerances of the tests above."""
    p = random_params(orc, 31)
    x, t = data(n, 32)
    mask = (np.random.default_rng(33).random((n, 2)) > 0.3).astype(np.float32)
    ctx.mlp_set(p)
    np.testing.assert_allclose(ctx.mlp_infer(x, mfma=False), orc.mlp_forward(p, x),
                               rtol=1e-4, atol=1e-5)
    loss, g = ctx.mlp_loss_grad(x, t, mask)
    ref_loss, ref_g = orc.mlp_loss_grad(p, x, t, mask)
    assert loss == pytest.approx(ref_loss, rel=1e-4)
    np.testing.assert_allclose(g, ref_g, rtol=2e-3, atol=2e-5)
