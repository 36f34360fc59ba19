"""A budget of learned iterations that the last allowed iteration uses up without convergence is reported as a fallback; one
that is not used up is not."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from dohp_amd.fields import lognormal_field  # noqa: E402
from dohp_amd.mesh import block_vertices, splitmix64_uniform  # noqa: E402


@pytest.mark.parametrize("mixed", [0, 1, 2])
def test_budget_used_up_at_the_iteration_limit(mixed):
    assert torch.cuda.is_available()
    import dohp_amd.capi as C
    M, p = (5, 4, 6), 4
    V = block_vertices(M, box=(0, 1, 0, 1, 0, 1), perturb=0.1, seed=3)
    fs = C.FS(M, p, V)
    op = C.Ellip(fs, p=2.0, kvert=lognormal_field(V, seed=7))
    plain = op.assemble_q1()
    op.set_q1_mode(1)
    q1 = op.assemble_q1()
    b = torch.as_tensor(2 * splitmix64_uniform(5, fs.nowned) - 1, dtype=torch.float64, device="cuda")
    for budget, max_it, fallback in ((3, 2, 0), (3, 3, 1), (3, 4, 1)):
        x = torch.zeros_like(b)
        st = op.solve(q1, b, x, mixed=mixed, rtol=1e-14, inner_rtol=1e-14, max_it=max_it, max_outer=1, fallback_q1=plain,
                      fallback_its=budget)
        assert (st["inner_its"], st["fallback"]) == (max_it, fallback), (budget, max_it)
