"""Block spaces with more lines or planes than a launch grid has blocks along y and z (65536)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from dohp_amd.mesh import block_vertices, splitmix64_uniform  # noqa: E402


@pytest.fixture(scope="module")
def C():
    assert torch.cuda.is_available()
    import dohp_amd.capi as capi
    return capi


def dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")


# four lines a block along y, eight planes a block along z; the last three at or just below the limit
@pytest.mark.parametrize("M", [(1, 262200, 1), (524300, 1, 1), (1, 262139, 1), (1, 262140, 1), (524279, 1, 1)])
def test_scatter(C, M):
    print(f"long box M={M}", flush=True)
    fs = C.FS(M, 1, block_vertices(M), dirichlet_mask=0)
    E = fs.element_nodes()
    xe = splitmix64_uniform(5, fs.nexpanded) - 0.5
    g0 = splitmix64_uniform(6, fs.nowned) - 0.5
    # a node has at most two elements: their sum is the same in either order, and g + x is added in the order of colours
    e = np.arange(fs.nelem) % 2
    for imode, start in ((C.INSERT_VALUES, np.zeros(fs.nowned)), (C.ADD_VALUES, g0)):
        ref = start.copy()
        for c in (0, 1):
            ref[E[e == c].reshape(-1)] += xe.reshape(fs.nelem, 8)[e == c].reshape(-1)
        g = dev(g0)
        fs.expanded_to_global(dev(xe), g, C.INHOMOGENEOUS, imode)
        np.testing.assert_array_equal(g.cpu().numpy(), ref)
