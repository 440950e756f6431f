"""Which kernel a call takes, where the rule can be asked without a device."""
import pytest

from fealpy_amd import _native as nat
from fealpy_amd import expr
from fealpy_amd.fem import integrators

ONE = 2.0 * expr.sin(expr.x) * expr.cos(expr.y) * expr.exp(expr.z)


@pytest.mark.parametrize("source,nq,n,one_pass", [
    (ONE, 4, 128, True), (expr.x + 1.0, 4, 40, True), (ONE, 4, 25, False), (ONE, 4, 6, False), (ONE, 20, 128, False),
    (ONE, 1, 128, False), (ONE + expr.x, 4, 128, False), (ONE + 0.5, 4, 10, False)])
def test_one_pass_load_vector_of_a_box(source, nq, n, one_pass):
    """Only one-term sources at the four-point rule on large grids: the others lost up to six times."""
    assert integrators._box_one_pass(source, nq, 6 * n ** 3) is one_pass


@pytest.mark.parametrize("points,ldof,sampled", [(7_680, 6, False), (490_000, 10, False), (1_200_000, 6, True),
                                                 (45_000, 20, True), (100_000, 35, True)])
def test_separable_coefficient_sampled_first(points, ldof, sampled):
    """A launch more only where it gains: small P2 assemblies lost a tenth by it."""
    assert integrators._sampled_first(points, ldof) is sampled


def test_sampling_no_cells_is_no_error():
    """The element tensors of no cells are formed from arrays without an address, as in fa_element_matrices."""
    L = nat.load()
    assert L.fa_sep_sample(3, 4, None, None, 0, None, None, None) == nat.FA_OK
    assert L.fa_sep_sample(3, 4, None, None, 1, None, None, None) == nat.FA_EINVAL
