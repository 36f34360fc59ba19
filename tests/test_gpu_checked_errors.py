"""A checked application that returns an error after its kernel was launched leaves nothing behind: the kernel, which met a
NaN, has ended when the call returns and cannot flag the next checked call."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from dohp_amd.mesh import block_vertices, splitmix64_uniform  # noqa: E402


def test_failed_call_does_not_flag_the_next():
    assert torch.cuda.is_available()
    import dohp_amd.capi as C
    M, p = (4, 5, 3), 3
    fs = C.FS(M, p, block_vertices(M))
    op = C.Ellip(fs, p=2.0)
    v = torch.as_tensor(splitmix64_uniform(6, fs.nowned), dtype=torch.float64, device="cuda")
    bad, y, z = v.clone(), torch.zeros_like(v), torch.zeros_like(v)
    bad[5] = float("nan")
    op.mat_mult_add(v, y)  # (tunes)
    w = torch.randn(4096, 4096, device="cuda")
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(3):
        with torch.cuda.stream(s):
            for _ in range(20):
                w = torch.tanh(w @ w)
        # an error of an earlier call of this thread, which the application finds after its launch
        assert C.lib().hipSetDevice(9999) != 0
        with pytest.raises(C.DohpError) as ei:
            op.mat_mult_add(bad, z, stream=s)
        assert ei.value.code == C.ERR_HIP
        assert s.query()  # (the call has waited for its stream)
        y.zero_()
        torch.cuda.synchronize()
        op.mat_mult_add(v, y, stream=s)
        assert torch.isfinite(y).all()
