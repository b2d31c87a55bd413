"""hexa20R element passes take two elements per wavefront: 1, 3 and 5 elements leave half a
wavefront empty in the last workgroup.  Same comparison and bounds as at the other tile edges
(1e-12 in FP64, 3e-6 in FP32 against the oracle's element matrices)."""

import pytest

pytest.importorskip("torch")
import test_gpu_pass_edges as edges  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("material", sorted(edges.PROPS))
@pytest.mark.parametrize("n", [(1, 1, 1), (3, 1, 1), (1, 5, 1)])
def test_hexa20r_odd_element_counts(material, n):
    edges.test_pass_and_assembly_at_tile_edges(material, "C3D20R", n)
