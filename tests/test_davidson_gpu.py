"""Davidson eigensolver with the diagonal and the learned (MLP) correction: the MLP oracle
pinned by finite differences, the GPU gradient kernels against it, diag(H) against the
assembled matrix, and Davidson energies against exact diagonalization and Lanczos."""
import numpy as np
import pytest

import dmrgpp_amd as dm
from dmrgpp_amd import problems
from oracle import mlp_oracle, oracle
from tests import fixtures


def _params(seed=3):
    rng = np.random.default_rng(seed)
    return rng.uniform(-0.4, 0.4, mlp_oracle.NPARAMS)


# ----------------------------------------------------------------------------- CPU tests


def test_mlp_oracle_gradient_matches_finite_differences():
    rng = np.random.default_rng(1)
    p = _params()
    x = rng.normal(size=(37, 4))
    t = rng.normal(size=37)
    g = mlp_oracle.gradient(p, x, t)
    idx = list(range(0, mlp_oracle.NPARAMS, 97)) + [mlp_oracle.OFF_B3, mlp_oracle.OFF_W3 + 5,
                                                   mlp_oracle.OFF_B1 + 7, mlp_oracle.OFF_B2 + 11]
    h = 1e-6
    for i in idx:
        e = np.zeros_like(p)
        e[i] = h
        fd = (mlp_oracle.loss(p + e, x, t) - mlp_oracle.loss(p - e, x, t)) / (2 * h)
        assert abs(fd - g[i]) < 1e-7 * max(1.0, abs(fd)), (i, fd, g[i])


def test_davidson_and_mlp_params_reject_bad_arguments():
    p = dm.davidson_params()
    assert p.tolerance == 1e-9 and p.precond == 1
    assert dm.lib().dmk_davidson_ground_d(None, None, None, None, None, None) == -1
    assert dm.lib().dmk_mlp_get_params(None, None) == -1


# ----------------------------------------------------------------------------- GPU tests


@pytest.mark.gpu
def test_gpu_mlp_forward_and_gradient_match_oracle():
    rng = np.random.default_rng(2)
    net = dm.Mlp(seed=5, capacity=1 << 12)
    p = _params(4).astype(np.float32)
    net.set_params(p)
    np.testing.assert_array_equal(net.params(), p)
    for count in (1, 63, 64, 1000, 20011):
        x = rng.normal(size=(count, 4)).astype(np.float32)
        t = rng.normal(size=count).astype(np.float32)
        y = net.forward(x)
        y_ref, _, _ = mlp_oracle.forward(p.astype(np.float64), x.astype(np.float64))
        assert np.abs(y - y_ref).max() < 1e-5 * max(1.0, np.abs(y_ref).max())
        g, loss = net.gradient(x, t)
        g_ref = mlp_oracle.gradient(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64))
        assert np.linalg.norm(g - g_ref) < 1e-5 * np.linalg.norm(g_ref), count
        assert abs(loss - mlp_oracle.loss(p, x, t)) < 1e-5 * mlp_oracle.loss(p, x, t)
    # Deterministic: the same batch gives bitwise the same gradient.
    g1, _ = net.gradient(x, t)
    g2, _ = net.gradient(x, t)
    np.testing.assert_array_equal(g1, g2)


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 15, 16, 17, 63, 64, 65, 768 * 64 - 1, 768 * 64, 768 * 64 + 17])
def test_gpu_mlp_forward_tiles(count):
    """Every remainder of a 16-sample tile, a wave, a workgroup and the whole grid."""
    rng = np.random.default_rng(count)
    net = dm.Mlp(seed=5, capacity=1)
    p = _params(rng).astype(np.float32)
    net.set_params(p)
    x = (3.0 * rng.standard_normal((count, 4))).astype(np.float32)
    x[0] = [np.inf, -np.inf, 0.0, 1.0] if count > 64 else x[0]
    y = net.forward(x)
    # FP32 bound: 8 roundings in layer 1, 70 in layer 2 and the output, 4 units per tanh (at
    # most 1); the split operands lose less than one more unit per product.
    u = 2.0 ** -24
    W1, b1, W2, b2, W3, b3 = mlp_oracle.unpack(p)
    f = x[1:] if count > 64 else x
    d1 = 8 * u * (np.abs(f.astype(np.float64)) @ np.abs(W1).T + np.abs(b1)) + 8 * u
    d2 = d1 @ np.abs(W2).T + 70 * u * (np.abs(W2).sum(axis=1) + np.abs(b2)) + 8 * u
    bound = d2 @ np.abs(W3) + 70 * u * (np.abs(W3).sum() + abs(b3))
    want = mlp_oracle.forward(p.astype(np.float64), f.astype(np.float64))[0]
    got = y[1:] if count > 64 else y
    assert np.all(np.abs(got - want) <= bound)
    if count > 64:  # a sample of infinities: what numpy makes of it, and no other sample's affair
        with np.errstate(invalid="ignore"):
            first = mlp_oracle.forward(p.astype(np.float64), x[:1].astype(np.float64))[0]
        assert np.isnan(first[0]) == np.isnan(y[0])
    net.close()


@pytest.mark.gpu
@pytest.mark.parametrize("lo,hi", [(2.0 ** -60, 1e-3), (1e-3, 0.5), (0.5, 0.999), (0.999, 1.001), (1.001, 3.0),
                                   (3.0, 20.0)])
def test_gpu_mlp_activation(lo, hi):
    """The activation on both sides of its line: layer 1's unit 0 is tanh(x0), which layer 2 keeps
    exactly apart from a power of two (its unit is 2^-40 times that, where tanh is the identity, and
    the smallest parts stay above FP32's smallest normal number).
    Odd to the last bit, and within 1.5 units in the last place of 64-bit tanh (tanhf: 1.34)."""
    n = 20000
    v = np.exp(np.random.default_rng(8).uniform(np.log(lo), np.log(hi), n)).astype(np.float32)
    x = np.zeros((2 * n, 4), dtype=np.float32)
    x[:n, 0], x[n:, 0] = v, -v
    p = np.zeros(mlp_oracle.NPARAMS, dtype=np.float32)
    p[0] = 1.0
    p[mlp_oracle.OFF_W2] = 2.0 ** -40
    p[mlp_oracle.OFF_W3] = 2.0 ** 40
    net = dm.Mlp(seed=5, capacity=1)
    net.set_params(p)
    y = net.forward(x)
    net.close()
    np.testing.assert_array_equal(y[n:], -y[:n])
    want = np.tanh(v.astype(np.float64))
    assert (np.abs(y[:n] - want) / np.spacing(want.astype(np.float32))).max() <= 1.5


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 17, 300])
def test_gpu_mlp_forward_infinite_and_largest_weights(count):
    """Weights at the ends of FP32: an infinity times 0 is NaN, opposite ones cancel to NaN, one alone
    saturates its unit, and the largest finite numbers multiply as they are."""
    x = np.random.default_rng(count).uniform(0.5, 1.5, (count, 4)).astype(np.float32)
    big = np.float32(np.finfo(np.float32).max)
    # Hidden units of layer 1: 0 is exactly 0, 1 positive, 2 its negative; layer 2 unit 0 takes them.
    for weights, want in (((np.inf, 0, 0), np.nan), ((0, np.inf, 0), 1.0), ((0, -np.inf, 0), -1.0),
                          ((0, np.inf, np.inf), np.nan), ((np.nan, 0, 0), np.nan),
                          ((big, 0, 0), 0.0), ((0, big, 0), 1.0), ((0, big, big), 0.0)):
        p = np.zeros(mlp_oracle.NPARAMS, dtype=np.float32)
        p[mlp_oracle.OFF_W1:mlp_oracle.OFF_B1].reshape(64, 4)[1:3, 0] = 1.0, -1.0
        p[mlp_oracle.OFF_W2:mlp_oracle.OFF_W2 + 3] = weights
        p[mlp_oracle.OFF_W3] = 1.0
        net = dm.Mlp(seed=5, capacity=1)
        net.set_params(p)
        np.testing.assert_array_equal(net.forward(x), np.full(count, want, dtype=np.float32))
        net.close()


@pytest.mark.gpu
@pytest.mark.parametrize("count", [1, 15, 65, 256 * 64, 256 * 64 + 1, 3 * 256 * 64 - 5])
def test_gpu_mlp_gradient_passes(count):
    """Remainders of a tile and a pass, and one, two and three passes per workgroup; the loss alone
    (after zero training steps) is the gradient call's."""
    rng = np.random.default_rng(count)
    net = dm.Mlp(seed=5, capacity=count)
    p = _params(rng).astype(np.float32)
    net.set_params(p)
    x = rng.standard_normal((count, 4)).astype(np.float32)
    t = rng.standard_normal(count).astype(np.float32)
    g, loss = net.gradient(x, t)
    want = mlp_oracle.gradient(p.astype(np.float64), x.astype(np.float64), t.astype(np.float64))
    # FP32 sums: about 300 roundings on the way to a term, and the partial sums' own.
    tol = 2.0 ** -24 * (300 + np.sqrt(count))
    assert np.linalg.norm(g - want) <= tol * np.linalg.norm(want)
    want_loss = mlp_oracle.loss(p, x, t)
    assert abs(loss - want_loss) <= tol * want_loss
    net.add_samples(x, t)
    _, alone = net.train(0, batch=count)
    assert abs(alone - want_loss) <= tol * want_loss
    net.close()


@pytest.mark.gpu
def test_gpu_mlp_training_reduces_loss():
    # Fit the clipped diagonal correction f3 = -f1 / f0 (a known function of the features).
    rng = np.random.default_rng(3)
    x = rng.normal(size=(32768, 4)).astype(np.float32)
    d = np.where(np.abs(x[:, 0]) < 0.05, np.sign(x[:, 0]) * 0.05 + (x[:, 0] == 0) * 0.05, x[:, 0])
    t = np.clip(-x[:, 1] / d, -10, 10).astype(np.float32)
    x[:, 3] = t
    net = dm.Mlp(seed=7, capacity=1 << 16)
    net.add_samples(x, t)
    assert net.samples() == x.shape[0]
    _, loss0 = net.gradient(x, t)
    last, after = net.train(iters=1500, batch=4096, lr=2e-3)
    assert after < 0.05 * loss0, (loss0, after)


def _dense_diag(prob):
    return np.diag(oracle.kron_form(prob))


@pytest.mark.gpu
def test_gpu_diagonal_matches_assembled_matrix():
    full, _, _, _ = fixtures.kron31_problem()
    prob = problems.random_problem([3, 5, 2, 7], [4, 1, 6, 3], nC=3, density=0.7, seed=9)
    for p in (full, prob):
        op = dm.BatchedGemm(p)
        d = dm.DeviceArray(p.n)
        op.diagonal(d)
        np.testing.assert_allclose(d.download(), _dense_diag(p), atol=1e-13)


@pytest.mark.gpu
@pytest.mark.parametrize("precond", ["none", "diag"])
def test_gpu_davidson_kron31_matches_ed(precond):
    full, _, _, _ = fixtures.kron31_problem()
    op = dm.BatchedGemm(full)
    init = dm.DeviceArray.from_host(np.random.default_rng(1234).uniform(-1, 1, full.n))
    z = dm.DeviceArray(full.n)
    r = op.davidson_ground(init, z, precond=precond, tolerance=1e-10, max_basis=12)
    assert r["converged"] == 1, r
    assert abs(r["energy"] - (-3.374932598687897)) < 1e-10
    assert r["residual"] < 1e-9
    zz = z.download()
    assert abs(np.linalg.norm(zz) - 1.0) < 1e-12


@pytest.mark.gpu
def test_gpu_davidson_matches_lanczos_on_qn_problem():
    left = problems.gaussian_histogram(160, 1.5, range(-3, 4))
    prob = problems.qn_problem(left, left, 0, problems.heisenberg_links(3), seed=4)
    op = dm.BatchedGemm(prob)
    init = dm.DeviceArray.from_host(np.random.default_rng(1234).uniform(-1, 1, prob.n))
    z = dm.DeviceArray(prob.n)
    lz = op.lanczos_ground(init, z, tolerance=0.0, stop_residual=1e-9, max_steps=400)
    dv = op.davidson_ground(init, z, precond="diag", tolerance=1e-9, max_basis=20)
    assert dv["converged"] == 1 and dv["residual"] < 2e-9
    assert lz["residual"] < 2e-9
    assert abs(dv["energy"] - lz["energy"]) < 1e-10 * abs(lz["energy"])


@pytest.mark.gpu
def test_gpu_learned_preconditioner_comparison():
    # Train on the first sweep of a Hubbard chain, then run the next sweep with plain Lanczos,
    # Davidson with the diagonal correction and Davidson with the network's own correction (no
    # fallback), all at FP64 residual 1e-9, each step from the same transformed wave function.
    # Equal energies; the network's matvec count is compared with the diagonal one directly.
    # The measured outcome is that the network does not gain: it needs 1.15x the diagonal
    # count here (1.14x on an 8x2 ladder and 1.22x on a 16x4 cylinder at m = 256), so the
    # assertion pins that it converges without costing more than 25 % extra matvecs, and that the
    # validation step, which decides from its own counts, keeps the diagonal method whenever
    # the network is not at least 5 % better on the validation superblocks.
    from dmrgpp_amd import learned

    out = learned.compare("hubbard-chain-12", train_sweeps=1, test_sweeps=1, train_iters=1500,
                          log=print)
    e = out["lanczos"]["energy"]
    for key in ("davidson-diag", "davidson-mlp", "davidson-learned"):
        assert abs(out[key]["energy"] - e) < 1e-9 * abs(e)
        assert out[key]["max_residual"] < 1.1e-9
    assert out["samples"] > 0 and out["loss"] < out["loss_untrained"]
    mlp, diag = out["davidson-mlp"]["matvecs"], out["davidson-diag"]["matvecs"]
    print(f"network / diagonal matvecs: {mlp} / {diag} = {mlp / diag:.3f}")
    assert mlp <= 1.25 * diag
    val = out["validation_matvecs"]
    assert out["chosen"] == ("mlp" if val["mlp"] < 0.95 * val["diag"] else "diag")
    assert out["lanczos"]["matvecs"] > diag


@pytest.mark.gpu
def test_gpu_superblock_compare_small():
    # The one-superblock comparison on a small Hubbard ladder superblock: Lanczos and Davidson
    # reach the FP64 residual at the same energy, and the mixed-precision ground states
    # (FP32 / BF16x3 with FP64 refinement) match FP64 Lanczos to 1e-10.
    from dmrgpp_amd import learned

    out = learned.superblock_compare("hubbard-ladder-8x2", at=5, log=lambda s: None)
    assert out["n"] > 10000 and out["npatches"] > 1
    e = out["lanczos"]["energy"]
    assert out["lanczos"]["residual"] < 1.1e-9 and out["davidson-diag"]["residual"] < 1.1e-9
    assert abs(out["davidson-diag"]["energy"] - e) < 1e-10 * abs(e)
    for prec in ("fp64", "fp32", "bf16x3"):
        assert out[prec]["ms_per_matvec"] > 0
        assert abs(out["ground_" + prec]["energy"] - e) < 1e-10 * abs(e)
