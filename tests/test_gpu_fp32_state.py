"""The FP32 copy of the linearization state (recomputing FP32 Jacobian, storage 0, checks off) under captured graphs and
on several streams: it belongs to the last residual, whoever evaluated or replayed that, and no application writes it."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from dohp_amd.mesh import block_vertices, splitmix64_uniform  # noqa: E402


@pytest.fixture(scope="module")
def C():
    assert torch.cuda.is_available()
    import dohp_amd.capi as capi
    return capi


class Problem:
    def __init__(self, C, M=(3, 2, 4), p=4):
        self.fs = C.FS(M, p, block_vertices(M, perturb=0.05, seed=2))
        self.op = C.Ellip(self.fs, p=1.5, eps=0.3, lam=0.4)
        self.op.set_storage(0)
        self.op.set_checks(0)
        n = self.fs.nowned
        new = lambda seed: torch.as_tensor(splitmix64_uniform(seed, n), dtype=torch.float64, device="cuda")
        self.u = [new(7), new(8), new(9)]
        self.v = 2 * new(6) - 1
        self.v32 = self.v.float()
        self.f = torch.zeros_like(self.v)
        # the reference action at each state in FP64, by an operator of its own
        op = C.Ellip(self.fs, p=1.5, eps=0.3, lam=0.4)
        self.ref = []
        for u in self.u:
            y = torch.zeros_like(self.v)
            op.function(u, self.f)
            op.mat_mult(self.v, y)
            self.ref.append(y)

    def check(self, y32, k):
        # state, contractions and physics in FP32: a few hundred roundings of 6e-8
        ref = self.ref[k]
        assert float(torch.linalg.norm(y32.double() - ref)) <= 1e-4 * float(torch.linalg.norm(ref)), k


def test_replayed_application_takes_the_last_state(C):
    """Residual, warm-up application, capture of the application; then residuals at other states and replays."""
    pr = Problem(C)
    y = torch.zeros_like(pr.v32)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    pr.op.function(pr.u[0], pr.f, stream=s)
    pr.op.mat_mult_f32(pr.v32, y, stream=s)
    s.synchronize()
    pr.check(y, 0)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        pr.op.mat_mult_f32(pr.v32, y, stream=s)
    for k in (1, 2, 0, 1):
        pr.op.function(pr.u[k], pr.f, stream=s)
        s.synchronize()
        g.replay()
        torch.cuda.synchronize()
        pr.check(y, k)


def test_replayed_residual_sets_the_fp32_state(C):
    """A captured residual replayed with other values of its input, followed by eager applications."""
    pr = Problem(C)
    y = torch.zeros_like(pr.v32)
    u = pr.u[0].clone()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    pr.op.function(u, pr.f, stream=s)
    pr.op.mat_mult_f32(pr.v32, y, stream=s)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        pr.op.function(u, pr.f, stream=s)
    for k in (1, 2, 0, 1):
        u.copy_(pr.u[k])
        g.replay()
        torch.cuda.synchronize()
        pr.op.mat_mult_f32(pr.v32, y, stream=s)
        s.synchronize()
        pr.check(y, k)


def test_applications_on_two_streams_after_a_residual(C):
    """The first application after a residual waits behind other work on its stream; one on a second stream does not
    depend on it."""
    pr = Problem(C)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    ya, yb = torch.zeros_like(pr.v32), torch.zeros_like(pr.v32)
    pr.op.function(pr.u[0], pr.f)
    pr.op.mat_mult_f32(pr.v32, ya)  # (tunes)
    w = torch.randn(4096, 4096, device="cuda")
    for k in (1, 2, 0):
        pr.op.function(pr.u[k], pr.f)
        torch.cuda.synchronize()
        with torch.cuda.stream(a):
            for _ in range(20):
                w = torch.tanh(w @ w)
        pr.op.mat_mult_f32(pr.v32, ya, stream=a)
        pr.op.mat_mult_f32(pr.v32, yb, stream=b)
        torch.cuda.synchronize()
        pr.check(ya, k)
        pr.check(yb, k)
