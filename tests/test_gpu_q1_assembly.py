"""The embedded-Q1 assembly's two kernels at their edges: every degree (elements per workgroup, rounds of sub-cells, LDS
size), partly filled workgroups, the three exponent paths, free boundaries, the ring of sub-cell layers over several
passes, and one matrix object refilled by operators of different degrees."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from dohp_amd.mesh import block_vertices, splitmix64_uniform  # noqa: E402
from oracle import oracle as O  # noqa: E402


@pytest.fixture(scope="module")
def C():
    assert torch.cuda.is_available()
    import dohp_amd.capi as capi
    return capi


def dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda")


def _pair(C, M, deg, mask, **prm):
    V = block_vertices(M, perturb=0.08, seed=4)
    fs, S = C.FS(M, deg, V, dirichlet_mask=mask), O.BlockSpace(M, deg, V, dirichlet_mask=mask)
    E, op = O.Ellip(S, exact=-1, **prm), C.Ellip(fs, **prm)
    uc = 0.3 * (2 * splitmix64_uniform(21, fs.nclosure) - 1)
    fs.dirichlet_commit(uc[fs.nowned:])
    return fs, op, E, uc


# The oracle sums the same terms in the reference's order: about a hundred roundings of 1.1e-16 of the largest ones.
@pytest.mark.parametrize("M,p,mask,ep,lam", [((1, 1, 1), 1, 0, 1.5, 0.0), ((5, 6, 9), 1, 7, 1.5, 0.7), ((3, 4, 3), 2, 6, 1.6, 0.0),
                                             ((3, 3, 2), 3, 7, 1.5, 0.3), ((2, 3, 1), 4, 1, 2.0, 0.0), ((1, 2, 3), 5, 0, 1.5, 0.0),
                                             ((2, 1, 2), 6, 7, 1.75, 0.2), ((1, 2, 1), 7, 6, 1.5, 0.0), ((2, 1, 1), 8, 7, 1.6, 0.3),
                                             ((1, 1, 2), 9, 0, 2.0, 0.4), ((1, 1, 1), 10, 6, 1.5, 0.1)])
def test_every_degree_matches_the_oracle(C, M, p, mask, ep, lam):
    print(f"q1 M={M} p={p} mask={mask} ep={ep} lam={lam}", flush=True)
    fs, op, E, uc = _pair(C, M, p, mask, p=ep, eps=0.5, lam=lam)
    A, R = op.assemble_q1(dev(uc[:fs.nowned])).to_scipy(), E.q1_matrix(uc)
    assert A.shape == R.shape
    d = np.abs((A - R).toarray()).max()
    assert d <= 1e-12 * np.abs(R.toarray()).max()
    assert (A != A.T).nnz == 0  # bitwise symmetric


def test_one_matrix_for_two_degrees(C):
    """Spaces with the same rows (11^3) and different degrees take the same matrix object in turn."""
    a = _pair(C, (6, 6, 6), 2, 7, p=1.5, eps=0.5)
    b = _pair(C, (4, 4, 4), 3, 7, p=1.5, eps=0.5)
    assert a[0].nowned == b[0].nowned
    mat = None
    for fs, op, E, uc in (a, b, a):
        mat = op.assemble_q1(dev(uc[:fs.nowned]), mat=mat)
        R = E.q1_matrix(uc)
        assert abs(mat.to_scipy() - R).max() <= 1e-12 * abs(R).max()


def test_several_passes(C):
    """A uniform mesh whose sub-cell matrices (288 bytes each) need three passes: the stencil of the corrected matrix
    repeats with the degree along the first direction, also across the passes' boundaries."""
    M, p = (48, 64, 64), 2
    fs = C.FS(M, p, block_vertices(M, box=(0, 1, 0, 1, 0, 1)))
    op = C.Ellip(fs, p=2.0)
    op.set_q1_mode(1)
    q1 = op.assemble_q1()
    mg = C.MG(q1)
    box, st = mg.level(0)
    st = torch.as_tensor(st).reshape(27, *box)
    assert box == (95, 127, 127)
    big = float(st.abs().max())
    inner = st[:, 1:-1]  # rows next to the boundary have dropped entries
    assert float((inner[:, p:] - inner[:, :-p]).abs().max()) <= 1e-13 * big
    for s in range(13):  # lower entries are the upper ones of the neighbours' rows
        di, dj, dk = s // 9 - 1, s // 3 % 3 - 1, s % 3 - 1
        a = st[s][max(0, -di):box[0] - max(0, di), max(0, -dj):box[1] - max(0, dj), max(0, -dk):box[2] - max(0, dk)]
        b = st[26 - s][max(0, di):box[0] + min(0, di), max(0, dj):box[1] + min(0, dj), max(0, dk):box[2] + min(0, dk)]
        assert torch.equal(a, b)
    ones = torch.ones(q1.nrows, dtype=torch.float64, device="cuda")
    y = torch.zeros_like(ones)
    q1.mult(ones, y)
    assert float(y.reshape(box)[1:-1, 1:-1, 1:-1].abs().max()) <= 1e-12 * big
