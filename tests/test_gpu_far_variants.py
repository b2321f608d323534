"""The far loop's variants at the edges of their ranges.

far_variant picks the short sine polynomials up to a phase of 0.32 inside a
panel, the long ones up to half a period, and the general form beyond that,
for a beta with a real part and for vanishing k.  Each side of each edge is
compared with the CPU oracle on the far entries alone (the near and diagonal
entries, which other kernels write, dominate the Frobenius norm).  Bound: the
phase k r <= 60 is rounded once on either side (60 * 2^-53 = 7e-15), the
13-point sums to a few 1e-16.
"""

import numpy as np
import pytest

import oracle
import sonium_amd as sa
from sonium_amd.mesh import ellipsoid, icosphere

from helpers import rel_fro

pytestmark = pytest.mark.gpu

TOL = 3e-14


def _radius(m):
    p = m.nodes[m.triangles]
    return np.max(np.linalg.norm(p - p.mean(axis=1, keepdims=True), axis=2))


def _far(m):
    c, _, area = m.element_geometry()
    return np.linalg.norm(c[:, None] - c[None], axis=2) / np.sqrt(area)[None] >= 3.0


def _cases():
    m = icosphere(1.0, 1)
    for phase in (0.01, 0.319, 0.321, 1.569, 1.571, 4.0):
        k = phase / 0.86 / _radius(m)
        yield k, 1j / k
        yield k, 0.3 - 0.2j
    yield 1.0, 0j
    yield 1e-45, 0.1j
    yield 1e-3, 0.1j


def _mixed(n):
    rng = np.random.default_rng(5)
    bt = (rng.random(n) < 0.3).astype(np.int32)
    adm = np.where((bt == 0) & (rng.random(n) < 0.5), 0.01 * (rng.standard_normal(n) + 1j), np.nan)
    return {"bc_type": bt, "admittance": adm}


@pytest.mark.parametrize("general", [False, True], ids=["rigid", "mixed"])
@pytest.mark.parametrize("k,beta", list(_cases()))
def test_far_entries_match_the_oracle(ctx, k, beta, general):
    m = icosphere(1.0, 1)
    bc = _mixed(m.num_elements) if general else {}
    ph = sa.PhysicsParams.from_wavenumber(k)
    tm = sa.TbemMesh(ctx, m, **bc)
    A = sa.build_tbem_system_with_beta(ctx, tm, ph, beta).matrix
    Ar, _ = oracle.build_tbem_system(m.nodes, m.triangles, k, beta, **bc)
    far = _far(m)
    assert rel_fro(A[far], Ar[far]) <= TOL
    assert rel_fro(A, Ar) <= 1e-12
    # the matrix-free product evaluates the same entries
    ws = sa.TbemAssemblyWorkspace(ctx, tm)
    x = np.random.default_rng(6).standard_normal((2, m.num_elements)) @ np.eye(m.num_elements)
    x = x[0] + 1j * x[1]
    y = sa.TbemExactOperator(ws, ph, beta).apply(x)
    ref = A @ x
    assert np.max(np.abs(y - ref)) <= 1e-13 * np.max(np.abs(A) @ np.abs(x))


@pytest.mark.parametrize("phase", [0.319, 0.321, 1.569, 1.571])
def test_batch_takes_the_single_system_variant(ctx, phase):
    """The batch assembly chooses per instance and gives the single system's bits."""
    meshes = [icosphere(1.0, 1), ellipsoid([1.3, 0.7, 0.6], 2)]
    ks = [phase / 0.86 / _radius(m) for m in meshes]
    tms = [sa.TbemMesh(ctx, m) for m in meshes]
    b = sa.Batch(ctx, tms)
    for betas in (None, [0.1 + 0.2j, 0.3j]):
        b.set_problem(ks, [np.array([[0.0, 0.0, 1.0]])] * 2, betas=betas)
        b.assemble()
        for i, (tm, k) in enumerate(zip(tms, ks)):
            ph = sa.PhysicsParams.from_wavenumber(k)
            beta = ph.burton_miller_beta() if betas is None else betas[i]
            assert np.array_equal(b.matrix(i), sa.build_tbem_system_with_beta(ctx, tm, ph, beta).matrix)


@pytest.mark.parametrize("general", [False, True], ids=["rigid", "mixed"])
@pytest.mark.parametrize("k,beta", list(_cases()))
def test_far_derivatives_match_the_oracle(ctx, k, beta, general):
    """d/dp with dk/dp = 0.7 and an unrelated beta derivative; the imaginary
    beta of half the cases also meets a beta derivative with a real part,
    which takes the general form."""
    m = icosphere(1.0, 1)
    bc = _mixed(m.num_elements) if general else {}
    ph = sa.PhysicsParams.from_wavenumber(k)
    ws = sa.TbemAssemblyWorkspace(ctx, sa.TbemMesh(ctx, m, **bc))
    far = _far(m)
    for beta_d in (-0.4j, 0.2 - 0.1j):
        A = ws.assemble_parameter_derivative(ph, beta, beta_d, sign=-1.0, wavenumber_scale=0.7,
                                             pressure_factor_derivative=3.0, admittance_scale=0.5).matrix
        Ar, _ = oracle.build_tbem_derivative(m.nodes, m.triangles, k, beta, beta_d, sign=-1.0, wavenumber_scale=0.7,
                                             pressure_factor_derivative=3.0,
                                             admittance_scale=0.5, **bc)
        assert rel_fro(A[far], Ar[far]) <= TOL
        assert rel_fro(A, Ar) <= 1e-12


@pytest.mark.parametrize("derivative", [False, True])
@pytest.mark.parametrize("axes,level,k", [((1.0, 1.0, 1.0), 0, 0.7), ((1.0, 1.0, 1.0), 2, 2.0),
                                          ((1.4, 0.35, 0.3), 2, 3.0), ((1.4, 0.35, 0.3), 3, 40.0)])
def test_near_entries_match_the_oracle(ctx, axes, level, k, derivative):
    """Subdivided pairs alone: one workgroup's worth of pairs and many, panels
    of aspect up to 5 (deep trees, up to the 110-leaf cap), the general form.
    The oracle forms positions before subtracting: 2^-53 * 1.4 over a leaf
    distance of at least 0.02, up to three powers of 1/r: 3e-14."""
    m = ellipsoid(axes, level)
    near = ~_far(m) & ~np.eye(m.num_elements, dtype=bool)
    ph = sa.PhysicsParams.from_wavenumber(k)
    for general in (False, True):
        bc = _mixed(m.num_elements) if general else {}
        ws = sa.TbemAssemblyWorkspace(ctx, sa.TbemMesh(ctx, m, **bc))
        if derivative:
            A = ws.assemble_parameter_derivative(ph, 1j / k, -1j / k ** 2).matrix
            Ar, _ = oracle.build_tbem_derivative(m.nodes, m.triangles, k, 1j / k, -1j / k ** 2, **bc)
        else:
            A = ws.assemble(ph, 1j / k).matrix
            Ar, _ = oracle.build_tbem_system(m.nodes, m.triangles, k, 1j / k, **bc)
        assert rel_fro(A[near], Ar[near]) <= 1e-13
