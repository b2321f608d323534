"""GPU tests of the warm-start MLP kernels.

* loss and every parameter gradient of the HIP forward/backward pass agree
  with the CPU oracle (oracle/mlp.py, BF16 rounding at the same points;
  tolerance 2e-2 relative Frobenius per layer block for the FP32 accumulation
  order and the BF16 flips it causes);
* predictions agree with the oracle;
* training on a smooth synthetic target lowers the loss by 10x;
* on a small frequency sweep the trained network's guesses lower the mean
  GMRES iteration count on held-out wavenumbers, with every solve converged
  on the recomputed FP64 residual (the learned-warm-start gain).
"""

import numpy as np
import pytest

import sonium_amd as sa
from oracle import mlp as omlp
from sonium_amd import warmstart as ws
from sonium_amd.mesh import icosphere

from helpers import rel_fro

pytestmark = pytest.mark.gpu


def _raw(rng, m):
    c = rng.standard_normal((m, 3))
    c /= np.linalg.norm(c, axis=1, keepdims=True)
    d = rng.standard_normal((m, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    k = rng.uniform(1, 12, size=(m, 1))
    return np.concatenate([c, c, d, k], axis=1).astype(np.float32)


def _blocks(width):
    off = 0
    for rows, cols in omlp.layer_shapes(width):
        yield off, rows * cols
        off += rows * cols
        yield off, rows
        off += rows


def test_gradients_match_oracle(ctx):
    net = ws.WarmStartMLP(ctx, width=512, seed=11)
    rng = np.random.default_rng(1)
    raw = _raw(rng, 512)
    t = rng.standard_normal((512, 2)).astype(np.float32)
    loss, g = net.loss_and_gradients(raw, t)
    p = net.params().astype(np.float64)
    loss_ref, g_ref, _ = omlp.loss_and_gradients(p, 512, raw, t, bf16_storage=True)
    assert abs(loss - loss_ref) <= 1e-4 * abs(loss_ref)
    for off, cnt in _blocks(512):
        a, b = g[off: off + cnt], g_ref[off: off + cnt]
        assert rel_fro(a, b) < 2e-2, (off, cnt, rel_fro(a, b))


def test_predictions_match_oracle(ctx):
    net = ws.WarmStartMLP(ctx, width=512, seed=12)
    rng = np.random.default_rng(2)
    raw = _raw(rng, 1000)
    y = net.predict(raw)
    y_ref = omlp.predict(net.params().astype(np.float64), 512, raw)
    assert rel_fro(y, y_ref) < 1e-2


@pytest.mark.parametrize("width", [64, 512, 1024, 2048])
def test_fused_inference_equals_layered_forward(ctx, width):
    """The fused inference kernel (all layers per 32-sample workgroup,
    activations in LDS) gives the layer-by-layer forward pass of training bit
    for bit, on ragged sample counts and after training steps; widths above
    1024 take the layered path."""
    net = ws.WarmStartMLP(ctx, width=width, seed=21)
    rng = np.random.default_rng(4)
    for m in (1, 257, 3000):
        raw = _raw(rng, m)
        assert np.array_equal(net.predict(raw), net.predict_layered(raw))
    net.set_dataset(_raw(rng, 4096), rng.standard_normal((4096, 2)).astype(np.float32))
    net.train(5, batch=1024)
    raw = _raw(rng, 777)
    assert np.array_equal(net.predict(raw), net.predict_layered(raw))
    net.close()


def test_training_lowers_loss(ctx):
    net = ws.WarmStartMLP(ctx, width=512, seed=13)
    rng = np.random.default_rng(3)
    raw = _raw(rng, 1 << 15)
    dc = (raw[:, 0:3] * raw[:, 6:9]).sum(1)
    k = raw[:, 9]
    t = np.stack([np.cos(0.3 * k * dc), np.sin(0.2 * k) * dc], axis=1).astype(np.float32)
    net.set_dataset(raw, t)
    losses = net.train(600, batch=4096, lr_max=2e-3, lr_min=1e-4, seed=3)
    assert np.all(np.isfinite(losses))
    assert losses[-20:].mean() < 0.1 * losses[:5].mean(), (losses[:5], losses[-20:])


def test_learned_warm_start_lowers_iterations(ctx):
    m = icosphere(1.0, 3)
    tm = sa.TbemMesh(ctx, m)
    c, n, _ = tm.geometry()
    wsp = sa.TbemAssemblyWorkspace(ctx, tm)
    d = np.array([0.0, 0.0, 1.0])
    ks = np.linspace(1.0, 4.0, 49)
    cfg = sa.GmresConfig(max_iterations=10, restart=100, tolerance=1e-8)
    sols, inputs, targets = {}, [], []
    for i, k in enumerate(ks):
        ph = sa.PhysicsParams.from_wavenumber(k)
        beta = ph.burton_miller_beta()
        system = wsp.assemble(ph, beta)
        b = sa.IncidentField([d]).compute_rhs_with_beta(tm, ph, beta)
        op = sa.DenseMatrixOperator(system)
        sol = sa.gmres(op, b, cfg)
        assert sol.converged
        sols[i] = (op, b, sol)
        if i % 2 == 0:
            inputs.append(ws.panel_inputs(c, n, k, d))
            targets.append(ws.density_to_target(sol.x, c, k, d))
    net = ws.WarmStartMLP(ctx, width=512, seed=5)
    net.set_dataset(np.concatenate(inputs), np.concatenate(targets))
    losses = net.train(800, batch=8192, lr_max=2e-3, lr_min=5e-5, seed=5)
    zero, learned = [], []
    for i in range(1, len(ks), 2):
        op, b, sol = sols[i]
        x0 = net.guess(c, n, ks[i], d)
        s2, used = ws.solve_with_guess(op, b, x0, cfg)
        assert s2.converged and s2.residual < 1e-8
        assert np.linalg.norm(b - op.apply(s2.x)) / np.linalg.norm(b) < 1e-8
        zero.append(sol.iterations)
        learned.append(s2.iterations)
    print("final loss", losses[-1], "zero-guess iterations", np.mean(zero), "learned", np.mean(learned))
    assert np.mean(learned) < np.mean(zero)


@pytest.mark.parametrize("width,m", [(64, 256), (192, 768), (128, 4352), (512, 256), (512, 12544), (1088, 512)])
def test_gradients_match_oracle_at_tile_edges(ctx, width, m):
    """Both product tiles (64 and 128 a side), mixed ones (a width of 64 times an
    odd number), one K slice and a short last slice: bounds of test_gradients_match_oracle."""
    net = ws.WarmStartMLP(ctx, width=width, seed=31)
    rng = np.random.default_rng(width + m)
    raw = _raw(rng, m)
    t = rng.standard_normal((m, 2)).astype(np.float32)
    loss, g = net.loss_and_gradients(raw, t)
    loss_ref, g_ref, _ = omlp.loss_and_gradients(net.params().astype(np.float64), width, raw, t, bf16_storage=True)
    assert abs(loss - loss_ref) <= 1e-4 * abs(loss_ref)
    for off, cnt in _blocks(width):
        assert rel_fro(g[off: off + cnt], g_ref[off: off + cnt]) < 2e-2, (off, cnt)


def _sample_indices(seed, step, batch, count):
    with np.errstate(over="ignore"):
        z = np.uint64(seed * 0x100000001B3 + step) + np.uint64(0x9E3779B97F4A7C15) * np.arange(1, batch + 1,
                                                                                              dtype=np.uint64)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return ((z ^ (z >> np.uint64(31))) % np.uint64(count)).astype(np.int64)


@pytest.mark.parametrize("width,batch", [(64, 256), (192, 1280), (512, 8192)])
def test_training_steps_are_adam_on_the_drawn_samples(ctx, width, batch):
    """Two one-step runs of train() against Adam in numpy on the gradients that
    loss_and_gradients gives for the same samples at the network's own
    parameters (so both round the same weights to BF16), and the refreshed
    BF16 copies against those that set_params makes.  Bound: the FP32 value of
    1 - 0.999^t is off by 6e-8 / 1e-3, 3e-5 of a step of lr; a few ulp of the
    parameters."""
    rng = np.random.default_rng(9)
    raw, t = _raw(rng, 3000), rng.standard_normal((3000, 2)).astype(np.float32)
    net = ws.WarmStartMLP(ctx, width=width, seed=8)
    ref = ws.WarmStartMLP(ctx, width=width, seed=8)
    net.set_dataset(raw, t)
    m1 = m2 = 0.0
    for step in range(2):
        p = net.params()
        losses = net.train(1, batch=batch, lr_max=1e-3, lr_min=1e-3, seed=4)
        at = _sample_indices(4, step, batch, 3000)
        ref.set_params(p)
        loss, g = ref.loss_and_gradients(raw[at], t[at])
        assert abs(losses[0] - loss) <= 1e-5 * loss
        g = g.astype(np.float64)
        m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
        want = p - 1e-3 * (m1 / (1 - 0.9 ** (step + 1))) / (np.sqrt(m2 / (1 - 0.999 ** (step + 1))) + 1e-8)
        q = net.params()
        assert np.max(np.abs(q - want)) <= 1e-3 * 1e-4 + 4e-7 * np.max(np.abs(p))
    ref.set_params(q)
    assert np.array_equal(net.predict(raw[:700]), ref.predict(raw[:700]))


def test_losses_of_long_runs_all_come_back(ctx):
    """The loss partials stay on the device for a bounded run of steps between reads."""
    rng = np.random.default_rng(10)
    raw = _raw(rng, 2000)
    net = ws.WarmStartMLP(ctx, width=64, seed=8)
    net.set_dataset(raw, raw[:, 0:2])
    losses = net.train(600, batch=512, seed=2)
    assert np.all(losses > 0) and losses[-50:].mean() < 0.2 * losses[:5].mean()
