"""sfx_get_layout describes what the forward steps read: on 2-D elastic meshes
the default and the gather scatter step on patches (control nodes, one kappa and
mu per element, points renumbered), the atomic one on per-point arrays."""
import numpy as np
import pytest


def _layout(scatter, per_point, host_only):
    from specfempp_amd import Engine2D, meshes

    n, h = 6, 20.0
    mesh = meshes.quad_mesh(n, n, 0.0, n * h, 0.0, n * h, materials=[meshes.elastic(2000.0, 3000.0, 1700.0)])
    c = mesh.coorg.copy()
    iz, ix = np.divmod(np.arange(c.shape[1]), n + 1)
    inner = (ix > 0) & (ix < n) & (iz > 0) & (iz < n)
    c[:, inner] += np.random.default_rng(3).uniform(-2.0, 2.0, size=(2, inner.sum()))
    mesh.coorg = c
    e = Engine2D(mesh, [], [], 1e-3, 4, 1, (), scatter=scatter, host_only=host_only)
    if per_point:
        shape = (mesh.nspec, 5, 5)
        mu = 5e9 * (1.0 + 0.01 * np.arange(25).reshape(5, 5)) * np.ones(shape)
        e.set_properties(*(x.astype(np.float32) for x in (2000.0 * np.ones(shape), 1e10 * np.ones(shape), mu)))
    lay = e.layout()
    e.close()
    return lay["geometry"], lay["element_properties"], lay["scatter"], lay["row_order"]


@pytest.mark.parametrize("host_only", [True, pytest.param(False, marks=pytest.mark.gpu)])
@pytest.mark.parametrize("scatter", ["colored", "gather"])
def test_layout_of_patches(scatter, host_only):
    assert _layout(scatter, False, host_only) == ("control_nodes_4", True, scatter, True)
    if not host_only:
        assert _layout(scatter, True, host_only) == ("control_nodes_4", False, scatter, True)


@pytest.mark.parametrize("host_only", [True, pytest.param(False, marks=pytest.mark.gpu)])
def test_layout_of_the_atomic_scatter(host_only):
    assert _layout("atomic", False, host_only) == ("point", False, "atomic", False)
