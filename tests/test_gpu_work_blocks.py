"""Work blocks of the solvers: kept for the next call, never mistaken for it.

A block that a call gives back is handed to the next one with its old contents,
on any thread, context or stream.  The answers may depend on neither: equal
bits whatever the idle blocks were filled with, and equal bits from threads
that exchange blocks while one of them captures a graph.
"""

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import sonium_amd as sa
from sonium_amd.mesh import icosphere
from sonium_amd.warmstart import WarmStartMLP

pytestmark = pytest.mark.gpu


class Problem:
    def __init__(self, level, k=1.7):
        self.ctx = sa.Context(0)
        self.mesh = sa.TbemMesh(self.ctx, icosphere(1.0, level))
        ph = sa.PhysicsParams.from_wavenumber(k)
        beta = ph.burton_miller_beta()
        self.system = sa.TbemAssemblyWorkspace(self.ctx, self.mesh).assemble(ph, beta)
        sa.IncidentField.plane_wave_z().add_to_system(self.system, self.mesh, ph, beta)
        self.op = sa.DenseMatrixOperator(self.system)
        self.lp = sa.LowpMatrix(self.system, "fp16")
        n = self.op.num_rows()
        rng = np.random.default_rng(n)
        self.b = np.asarray(self.system.rhs)
        self.B = rng.standard_normal((n, 5)) + 1j * rng.standard_normal((n, 5))
        self.batch = sa.Batch(self.ctx, [self.mesh] * 2)
        self.batch.set_problem([k, 1.1 * k], [[(0.0, 0.0, 1.0)]] * 2)
        self.batch.assemble()

    def answers(self):
        b, B = self.b, self.B
        plain = sa.GmresConfig(max_iterations=4, restart=30, tolerance=1e-8)
        block = sa.BlockGmresConfig(max_iterations=4, restart=30, tolerance=1e-8)
        ir = sa.GmresIrConfig(max_outer_iterations=6, outer_tolerance=1e-8, max_inner_iterations=20)
        out = [sa.gmres(self.op, b, plain).x, sa.block_gmres(self.op, B, block).x,
               sa.gmres_ir(self.op, self.lp, B, ir)[0], self.op.apply(b)]
        self.batch.solve("fp64", restart=20, max_cycles=4, tolerance=1e-8, use_graph=True)
        return [np.asarray(x) for x in out + list(self.batch.solutions())]


    def calls(self):
        """Every kind of call that takes work blocks, each from nothing but its inputs."""
        n, b, B = self.op.num_rows(), self.b, self.B
        rng = np.random.default_rng(n + 1)
        wide = rng.standard_normal((n, 40)) + 1j * rng.standard_normal((n, 40))
        low = rng.standard_normal((48, 24)) @ rng.standard_normal((24, 48))
        samples = rng.standard_normal((700, 10)).astype(np.float32)
        values = rng.standard_normal((700, 2)).astype(np.float32)
        points = 3.0 * rng.standard_normal((50, 3))
        ph = sa.PhysicsParams.from_wavenumber(1.7)
        field = sa.IncidentField.plane_wave_z()
        block = lambda restart, cycles=4: sa.BlockGmresConfig(max_iterations=cycles, restart=restart, tolerance=1e-8)
        ir = sa.GmresIrConfig(max_outer_iterations=6, outer_tolerance=1e-8, max_inner_iterations=20)

        def batch():
            self.batch.solve("fp64", restart=20, max_cycles=4, tolerance=1e-8, use_graph=True)
            return self.batch.solutions()

        def train():
            net = WarmStartMLP(self.ctx, width=128, seed=3)
            net.set_dataset(samples, values)
            out = [net.train(6, batch=512), net.params(), net.predict(samples), net.predict_layered(samples)]
            return out + [net.loss_and_gradients(samples[:256], values[:256])[1]]

        def recycled():
            sub = sa.GcroDrSubspace(self.ctx, n, 6)
            cfg = sa.GcroDrConfig(max_iterations=40, restart=12, tolerance=1e-8)
            return [sa.gcro_dr(self.op, v, None, sub, cfg).x for v in (b, B[:, 0])]

        def spent():  # a basis beyond its space: the least squares grow
            op = sa.CallbackOperator(self.ctx, 48, lambda x: low @ x)
            return [sa.block_gmres(op, wide[:48, :3], block(30, 1)).x]

        return {
            "gmres": lambda: [sa.gmres(self.op, b, sa.GmresConfig(max_iterations=4, restart=30, tolerance=1e-8)).x],
            "gmres restarts": lambda: [sa.gmres(self.op, b, sa.GmresConfig(max_iterations=9, restart=4,
                                                                         tolerance=1e-8)).x],
            "block": lambda: [sa.block_gmres(self.op, B, block(30)).x],
            "wide block": lambda: [sa.block_gmres(self.op, wide, block(3)).x],
            "deflated block": lambda: [sa.block_gmres(self.op, np.concatenate([B, B[:, :2]], 1), block(30)).x],
            "spent block": spent,
            "columns": lambda: [sa.gmres_block(self.op, B, sa.GmresConfig(max_iterations=4, restart=9,
                                                                         tolerance=1e-8))[0]],
            "refinement": lambda: [sa.gmres_ir(self.op, self.lp, B, ir)[0], sa.gmres_ir(self.op, self.lp, wide, ir)[0]],
            "products": lambda: [self.op.apply(b), self.op.apply_block(wide), self.lp.apply(B)],
            "batch": batch,
            "recycled": recycled,
            "field": lambda: [sa.compute_scattered_field(points, self.mesh, b, ph)],
            "right-hand side": lambda: [field.compute_rhs_with_beta(self.mesh, ph, ph.burton_miller_beta())],
            "network": train,
        }


def test_answers_do_not_depend_on_what_a_block_held():
    """NaN, huge numbers (and as integers, minus one and far out of any range)
    and zeros in every idle block before each call."""
    p = Problem(2)
    calls = p.calls()
    want = {name: [np.array(x) for x in call()] for name, call in calls.items()}
    held = sa.live_device_bytes()
    for byte in (0xFF, 0x7F, 0x00):
        for name, call in calls.items():
            assert sa.debug_fill_idle_memory(byte) > 0
            for x, y in zip(call(), want[name]):
                assert np.array_equal(x, y) and np.all(np.isfinite(y)), (name, byte)
    assert sa.live_device_bytes() == held, "idle blocks belong to nobody"


def test_threads_that_exchange_blocks_match_serial_bits():
    problems = [Problem(1), Problem(2), Problem(2), Problem(3)]
    want = [p.answers() for p in problems]

    def work(i):
        return [problems[i].answers() for _ in range(3)]

    with ThreadPoolExecutor(len(problems)) as pool:
        got = list(pool.map(work, range(len(problems))))
    for runs, ref in zip(got, want):
        for run in runs:
            for x, y in zip(run, ref):
                assert np.array_equal(x, y)


def test_idle_blocks_are_given_back():
    p = Problem(2)
    want = p.answers()
    device, pinned = sa.trim_idle_memory()
    assert device > 0 and pinned > 0
    assert sa.trim_idle_memory() == (0, 0)
    for x, y in zip(p.answers(), want):
        assert np.array_equal(x, y)
    # a budget that idle blocks would exceed
    p.ctx.set_device_budget(p.ctx.device_budget()[1] + 1024)
    assert sa.trim_idle_memory()[0] == 0
    p.ctx.set_device_budget(0)
    p.answers()
    with pytest.raises(sa.SbhError, match="budget"):
        p.ctx.set_device_budget(p.ctx.device_budget()[1] + 1024)
        sa.TbemSystem(p.ctx, 1000)
    assert sa.trim_idle_memory()[0] == 0
