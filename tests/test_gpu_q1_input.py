"""The embedded-Q1 assembly has read its input vector when it returns: the caller may overwrite it on any stream, also
while the stream of the assembly is behind with other work."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from dohp_amd.mesh import block_vertices, splitmix64_uniform  # noqa: E402


def test_input_may_be_overwritten():
    assert torch.cuda.is_available()
    import dohp_amd.capi as C
    M, p = (3, 4, 2), 3
    fs = C.FS(M, p, block_vertices(M))
    op = C.Ellip(fs, p=1.5, eps=0.3)
    u = torch.as_tensor(splitmix64_uniform(7, fs.nowned), dtype=torch.float64, device="cuda")
    mat = op.assemble_q1(u)
    ref = mat.to_scipy()
    w = torch.randn(4096, 4096, device="cuda")
    s = torch.cuda.Stream()
    for _ in range(2):
        v = u.clone()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            for _ in range(20):
                w = torch.tanh(w @ w)
        op.assemble_q1(v, mat=mat, stream=s)
        v.fill_(float("nan"))
        torch.cuda.synchronize()
        assert abs(mat.to_scipy() - ref).max() == 0
