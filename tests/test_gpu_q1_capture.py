"""The embedded-Q1 assembly is refused in a graph capture, also where the matrix, its tables and workspace are there, and
the matrix keeps its values."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from dohp_amd.mesh import block_vertices, splitmix64_uniform  # noqa: E402


def test_reassembly_is_refused_in_a_capture():
    assert torch.cuda.is_available()
    import dohp_amd.capi as C
    M, p = (3, 4, 2), 3
    fs = C.FS(M, p, block_vertices(M))
    op = C.Ellip(fs, p=1.5, eps=0.3)
    u = torch.as_tensor(splitmix64_uniform(7, fs.nowned), dtype=torch.float64, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    mat = op.assemble_q1(u, stream=s)
    before = mat.to_scipy()
    g, t = torch.cuda.CUDAGraph(), torch.zeros(4, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        t += 1
        with pytest.raises(C.DohpError) as ei:
            op.assemble_q1(u + 0, mat=mat, stream=s)
        assert ei.value.code == C.ERR_HIP
    g.replay()
    torch.cuda.synchronize()
    assert abs(mat.to_scipy() - before).max() == 0
    assert float(t[0]) == 1
    again = op.assemble_q1(u, mat=mat, stream=s)
    s.synchronize()
    assert abs(again.to_scipy() - before).max() == 0
