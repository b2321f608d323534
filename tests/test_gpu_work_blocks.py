"""Work blocks of the solvers: kept for the next call, never mistaken for it.

A block that a call gives back is handed to the next one with its old contents,
on any thread, context or stream.  The answers may depend on neither: equal
bits whatever ran before, also after blocks were left full of NaN, and equal
bits from threads that exchange blocks while one of them captures a graph.
"""

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import sonium_amd as sa
from sonium_amd.mesh import icosphere

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

    def answers(self, b=None, B=None):
        b, B = self.b if b is None else b, self.B if B is None else B
        plain = sa.GmresConfig(max_iterations=4, restart=30, tolerance=1e-8)
        block = sa.BlockGmresConfig(max_iterations=4, restart=30, tolerance=1e-8)
        ir = sa.GmresIrConfig(max_outer_iterations=6, outer_tolerance=1e-8, max_inner_iterations=20)
        out = [sa.gmres(self.op, b, plain).x, sa.block_gmres(self.op, B, block).x,
               sa.gmres_ir(self.op, self.lp, B, ir)[0], self.op.apply(b)]
        self.batch.solve("fp64", restart=20, max_cycles=4, tolerance=1e-8, use_graph=True)
        return [np.asarray(x) for x in out + list(self.batch.solutions())]


def test_answers_do_not_depend_on_what_a_block_held():
    p = Problem(2)
    want = p.answers()
    held = sa.live_device_bytes()
    for value in (np.nan, np.inf, 1e300):
        try:
            p.answers(np.full_like(p.b, value), np.full_like(p.B, value))
        except sa.SbhError:
            pass
        for x, y in zip(p.answers(), want):
            assert np.array_equal(x, y)
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
