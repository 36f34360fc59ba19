"""Gathers and scatters of block spaces at their edges (sums bit for bit in the order of the element colours), the FP32
copy of the linearization state, and the non-finite flag of checked calls beside unchecked ones."""
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


@pytest.mark.parametrize("M,p,mask", [((1, 1, 1), 1, 0), ((2, 2, 2), 1, 7), ((1, 2, 3), 1, 6), ((2, 3, 4), 2, 7), ((3, 2, 5), 3, 1),
                                      ((5, 4, 17), 4, 2), ((2, 2, 2), 10, 4), ((1, 1, 2), 15, 0), ((4, 7, 9), 7, 7)])
def test_block_gather_and_scatter(C, M, p, mask):
    print(f"transfer M={M} p={p} mask={mask}", flush=True)
    fs = C.FS(M, p, block_vertices(M), dirichlet_mask=mask)
    E = fs.element_nodes()
    n3 = (p + 1) ** 3
    dv = splitmix64_uniform(3, fs.nclosure - fs.nowned) + 2
    fs.dirichlet_commit(dv)
    g = splitmix64_uniform(4, fs.nowned) - 0.5
    for hmode, edge in ((C.INHOMOGENEOUS, dv), (C.HOMOGENEOUS, 0 * dv)):
        ref = np.concatenate([g, edge])[E].reshape(-1)
        x = torch.full((fs.nexpanded + 4,), 5.0, dtype=torch.float64, device="cuda")
        fs.global_to_expanded(dev(g), x, hmode)
        np.testing.assert_array_equal(x[:-4].cpu().numpy(), ref)
        fs.global_to_expanded(dev(g), x, hmode, C.ADD_VALUES)
        np.testing.assert_array_equal(x.cpu().numpy(), np.concatenate([ref + ref, np.full(4, 5.0)]))
    xe = splitmix64_uniform(5, fs.nexpanded) - 0.5
    e = np.arange(fs.nelem)
    colour = ((e // (M[1] * M[2])) % 2) * 4 + ((e // M[2]) % M[1] % 2) * 2 + e % M[2] % 2
    for imode, start in ((C.INSERT_VALUES, np.zeros(fs.nclosure)), (C.ADD_VALUES, np.append(g, dv))):
        ref = start.copy()
        for c in range(8):
            for q in np.nonzero(colour == c)[0]:
                ref[E[q]] += xe[q * n3:(q + 1) * n3]
        gd = dev(g)
        fs.expanded_to_global(dev(xe), gd, C.INHOMOGENEOUS, imode)
        np.testing.assert_array_equal(gd.cpu().numpy(), ref[:fs.nowned])


def test_fp32_state_follows_the_residual(C):
    """Each residual's state reaches the recomputing FP32 Jacobian, also when FP64 applications came between."""
    M, p = (3, 2, 4), 4
    fs = C.FS(M, p, block_vertices(M, perturb=0.05, seed=2))
    op = C.Ellip(fs, p=1.5, eps=0.3, lam=0.4)
    op.set_storage(0)
    f, y = torch.zeros(fs.nowned, dtype=torch.float64, device="cuda"), torch.zeros(fs.nowned, dtype=torch.float64, device="cuda")
    v = dev(2 * splitmix64_uniform(6, fs.nowned) - 1)
    y32 = torch.zeros(fs.nowned, dtype=torch.float32, device="cuda")
    for seed in (7, 8, 9):
        op.function(dev(splitmix64_uniform(seed, fs.nowned)), f)
        op.mat_mult(v, y)
        op.mat_mult_f32(v.float(), y32)
        # state, contractions and physics in FP32: a few hundred roundings of 6e-8
        assert float(torch.linalg.norm(y32.double() - y)) <= 1e-4 * float(torch.linalg.norm(y))


def test_unchecked_nan_does_not_reach_a_checked_call(C):
    M, p = (6, 6, 6), 5
    fs = C.FS(M, p, block_vertices(M))
    op = C.Ellip(fs, p=2.0)
    v = dev(splitmix64_uniform(6, fs.nowned))
    bad, y, z = v.clone(), torch.zeros_like(v), torch.zeros_like(v)
    bad[5] = float("nan")
    op.mat_mult(v, y)
    for _ in range(5):
        op.set_checks(0)
        op.mat_mult(bad, z)
        op.set_checks(1)
        op.mat_mult(v, y)
        assert torch.isfinite(y).all()
        with pytest.raises(C.DohpError) as ei:
            op.mat_mult(bad, z)
        assert ei.value.code == C.ERR_NAN
