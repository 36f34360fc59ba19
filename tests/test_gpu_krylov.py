"""The fused conjugate gradients against the textbook recurrence in torch (the library's operator and V-cycle, every
scalar on the host): iterates after a few iterations, iteration limits, recorded iterates, one-unknown systems."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from dohp_amd.fields import lognormal_field  # noqa: E402
from dohp_amd.mesh import block_vertices, splitmix64_uniform  # noqa: E402


@pytest.fixture(scope="module")
def C():
    assert torch.cuda.is_available()
    import dohp_amd.capi as capi
    return capi


def _problem(C, M, p):
    V = block_vertices(M, box=(0, 1, 0, 1, 0, 1), perturb=0.1, seed=3)
    fs = C.FS(M, p, V)
    op = C.Ellip(fs, p=2.0, kvert=lognormal_field(V, seed=7))
    op.set_scatter(0)  # a fixed summation order: the two loops apply the same operator
    op.set_q1_mode(1)
    q1 = op.assemble_q1()
    b = torch.as_tensor(2 * splitmix64_uniform(5, fs.nowned) - 1, dtype=torch.float64, device="cuda")
    return op, q1, b


def _textbook(C, op, q1, b, mixed, its):
    """x_1..x_its of CG from zero; mixed = 2: flexible beta, the preconditioner applied in FP32."""
    mg = C.MG(q1, smooth_degree=1)
    x, r, z, q = torch.zeros_like(b), b.clone(), torch.empty_like(b), torch.empty_like(b)
    out = []

    def precondition():
        if mixed == 2:
            z32 = torch.empty(b.shape, dtype=torch.float32, device="cuda")
            mg.apply_f32(r.float(), z32)
            z.copy_(z32)
        else:
            mg.apply(r, z)

    precondition()
    p, rz = z.clone(), float(r @ z)
    for _ in range(its):
        op.mat_mult(p, q)
        alpha = rz / float(p @ q)
        x = x + alpha * p
        r = r - alpha * q
        out.append(x)
        precondition()
        rzn = float(r @ z)
        p = z + (-alpha * float(z @ q) / rz if mixed == 2 else rzn / rz) * p
        rz = rzn
    return out


# Sizes: one unknown, fewer unknowns than a reduction's blocks, more than its threads (2048 * 256), odd.  The two loops
# differ by the rounding of sums and scalars (1e-15 each); CG carries it on by a factor of a few per iteration: 1e-10.
@pytest.mark.parametrize("M,p", [((2, 2, 2), 1), ((2, 3, 4), 3), ((11, 13, 17), 6)])
@pytest.mark.parametrize("mixed", [0, 2])
def test_iterates_match_the_textbook(C, M, p, mixed):
    print(f"CG M={M} p={p} mixed={mixed}", flush=True)
    op, q1, b = _problem(C, M, p)
    n = b.numel()
    its = 1 if n == 1 else 6
    ref = _textbook(C, op, q1, b, mixed, its)
    for k in range(1, its + 1):
        x = torch.zeros_like(b)
        st = op.solve(q1, b, x, mixed=mixed, rtol=1e-14, max_it=k)
        assert st["inner_its"] == k
        assert float(torch.linalg.norm(x - ref[k - 1])) <= 1e-10 * float(torch.linalg.norm(ref[k - 1])), k
    x = torch.zeros_like(b)
    assert op.solve(q1, b, x, mixed=mixed, rtol=1e-10, max_it=0)["inner_its"] == 0 and not x.any()
    if mixed == 0 and n > 1:  # recorded iterates: every second one
        snap = torch.zeros(3, n, dtype=torch.float64, device="cuda")
        st = op.solve(q1, b, torch.zeros_like(b), rtol=1e-14, max_it=5, record=(snap, 2))
        assert st["nsnap"] == 2 and not snap[2].any()
        for i in (0, 1):
            assert float(torch.linalg.norm(snap[i] - ref[2 * i + 1])) <= 1e-10 * float(torch.linalg.norm(ref[2 * i + 1]))


def test_converged_start_and_repeat(C):
    """A start that already satisfies the tolerance takes no iteration; the next solve is not affected by the
    preconditioner application that the last iteration may have launched ahead."""
    op, q1, b = _problem(C, (3, 4, 5), 4)
    x = torch.zeros_like(b)
    first = op.solve(q1, b, x, mixed=2, rtol=1e-10)
    y = x.clone()
    assert op.solve(q1, b, y, mixed=2, rtol=1e-9)["inner_its"] == 0 and torch.equal(x, y)
    z = torch.zeros_like(b)
    again = op.solve(q1, b, z, mixed=2, rtol=1e-10)
    assert again["inner_its"] == first["inner_its"] and torch.equal(x, z)
    r = torch.zeros_like(b)
    op.mat_mult(x, r)
    assert float(torch.linalg.norm(b - r)) <= 2e-10 * float(torch.linalg.norm(b))
