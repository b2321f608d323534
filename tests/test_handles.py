"""Objects that the package hands to the library are of the kind that the call
takes: anything else is a TypeError before the library sees an address (no GPU
is needed, and none of these calls reaches the library)."""

import numpy as np
import pytest

import sonium_amd as sa
from sonium_amd.warmstart import WarmStartMLP


class _Impostor:
    """Has what the wrappers look at, and a handle of something else."""

    num_dofs = num_elements = num_rhs = 4
    length, ptr = 4, 0
    ctx = property(lambda self: self)

    def num_rows(self):
        return 4

    @property
    def handle(self):
        pytest.fail("the handle of another kind of object was taken")

    _h = handle


class _Operator(sa.DenseMatrixOperator):
    def num_rows(self):
        return 4


def _made(kind):
    return object.__new__(kind)  # of the right kind, without a handle


def _calls():
    other, b, B = _Impostor(), np.zeros(4, complex), np.zeros((4, 2), complex)
    ph, cfg = sa.PhysicsParams.from_wavenumber(1.0), sa.GmresConfig(max_iterations=1)
    batch = _made(sa.Batch)
    batch._h = None
    system = _made(sa.TbemSystem)
    system._h, system.num_dofs, system.ctx = None, 4, other
    op = _made(_Operator)
    op._h, op.system, op.ctx = None, system, other
    return {
        "vector": lambda: sa.DeviceVector(other, 4),
        "system": lambda: sa.TbemSystem(other, 4),
        "workspace": lambda: sa.TbemAssemblyWorkspace(other, other),
        "dense operator of an operator": lambda: sa.DenseMatrixOperator(op),
        "exact operator": lambda: sa.TbemExactOperator(other, ph),
        "low-precision copy of an operator": lambda: sa.LowpMatrix(op),
        "low-precision copy": lambda: sa.LowpMatrix(other),
        "jacobi of a system": lambda: sa.JacobiPreconditioner(other),
        "gmres": lambda: sa.gmres(other, b, cfg),
        "gmres preconditioner": lambda: sa.gmres_preconditioned_with_guess(op, other, b, None, cfg),
        "block": lambda: sa.block_gmres(other, B),
        "columns": lambda: sa.gmres_block(other, B, cfg),
        "refinement": lambda: sa.gmres_ir(op, other, B, sa.GmresIrConfig()),
        "batch": lambda: sa.Batch(_made_context(), [other]),
        "learned guesses": lambda: batch.learned_guesses(other),
        "network": lambda: WarmStartMLP(other),
    }


def _made_context():
    c = _made(sa.Context)
    c._h = None
    return c


@pytest.mark.parametrize("name", sorted(_calls()))
def test_another_kind_of_object_is_refused(name):
    with pytest.raises(TypeError, match="expected a"):
        _calls()[name]()


def test_kinds_that_share_an_interface_are_accepted():
    for kind in (sa.TbemExactOperator, sa.CallbackOperator, sa.DenseMatrixOperator):
        op = _made(kind)
        op._h = None
        assert sa._op_h(op) is None
    for kind in (sa.JacobiPreconditioner, sa.IdentityPreconditioner, sa.CallbackPreconditioner):
        pc = _made(kind)
        pc._h = None
        assert sa._precond_h(pc) is None
    assert sa._precond_h(None) is None
