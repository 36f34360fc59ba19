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


@pytest.mark.parametrize("M,p", [((65540, 1, 1), 1), ((32770, 1, 1), 2), ((1, 262200, 1), 1), ((1, 131100, 1), 2)])
def test_q1_assembly(C, M, p):
    """A uniform bar, corrected matrix: symmetric, and with free boundaries every row sums to zero; away from the ends the
    rows repeat with the degree."""
    print(f"long bar M={M} p={p}", flush=True)
    fs = C.FS(M, p, block_vertices(M, box=(0, M[0], 0, M[1], 0, M[2])), dirichlet_mask=0)
    op = C.Ellip(fs, p=2.0)
    op.set_q1_mode(1)
    A = op.assemble_q1().to_scipy()
    big = abs(A).max()
    # a row adds up to 27 entries of at most eight terms each: some hundred roundings of 1.1e-16
    assert np.abs(A.sum(axis=1)).max() <= 1e-13 * big
    assert (A != A.T).nnz == 0
    d = A.diagonal()
    cross = (p + 1) ** 2  # rows of a plane across a bar along x
    if M[0] > 1:
        d = d.reshape(-1, cross)
    else:  # node (i, j, k) of a bar along y
        d = d.reshape(p + 1, -1, p + 1).transpose(1, 0, 2).reshape(-1, cross)
    assert d.min() > 0
    inner = d[p:-p]
    assert np.abs(inner[p:] - inner[:-p]).max() <= 1e-13 * big
