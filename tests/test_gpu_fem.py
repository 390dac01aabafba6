"""GPU elastic tets (fem/fem.py:21-34,138-203; time_integrator_base.py:
124-137) against the oracle's per-thread restatement of tet_kernel_sparse:
rest shapes, triplet rows/cols and blocks bit-exact (the same operations in
the same order), per-tet energies within fp32 log rounding, forces within
the rounding of their float atomics; on the cube-drop cubes and on the
twisted rods' tets."""
import numpy as np
import pytest
import torch

from ipc_warp_amd import ops, scenes

pytestmark = pytest.mark.gpu

MU, LAM = 2.0e6, 2.0e7


def _case(name):
    if name == "cubes":
        soup = scenes.two_cubes_on_ground(seed=11, n=8, gap=4e-4, jitter=2e-4)
        rng = np.random.default_rng(5)
        x = soup.x + (1e-2 * rng.normal(size=soup.x.shape)).astype(np.float32)
        return soup.xcs, x.astype(np.float32), soup.tets
    soup, _, _ = scenes.rod_bundle(seed=0)
    T = soup.tets[:40000]
    return soup.xcs, soup.x, T


@pytest.mark.parametrize("name", ["cubes", "rods"])
def test_tet_kernels_match_oracle(dev, oracle, name):
    xcs, x, T = _case(name)
    T = np.ascontiguousarray(T, np.int32)
    n = T.shape[0]
    xcs_t, x_t, T_t = (torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in (xcs, x, T))
    Bm, W = ops.tet_rest(xcs_t, T_t)
    rBm, rW = oracle.tet_rest(xcs, T)
    torch.cuda.synchronize()
    assert np.array_equal(Bm.cpu().numpy().view(np.uint32), rBm.view(np.uint32))
    assert np.array_equal(W.cpu().numpy().view(np.uint32), rW.view(np.uint32))
    rows = torch.empty(16 * n, dtype=torch.int32, device=dev)
    cols = torch.empty_like(rows)
    vals = torch.empty((16 * n, 3, 3), dtype=torch.float32, device=dev)
    b = torch.zeros_like(x_t)
    ops.tet_hessian(x_t, T_t, Bm, W, MU, LAM, rows, cols, vals, b)
    psi = torch.empty(n, dtype=torch.float32, device=dev)
    e = torch.zeros(1, dtype=torch.float64, device=dev)
    ops.tet_energy(x_t, T_t, Bm, W, MU, LAM, psi, e)
    torch.cuda.synchronize()
    rr, rc, rv, rf = oracle.tet_hessian(x, T, rBm, rW, MU, LAM)
    assert np.array_equal(rows.cpu().numpy(), rr) and np.array_equal(cols.cpu().numpy(), rc)
    assert np.array_equal(vals.cpu().numpy().view(np.uint32), rv.view(np.uint32))
    gf = b.cpu().numpy()
    assert np.abs(gf - rf).max() <= 1e-5 * np.abs(rf).max()
    rpsi = oracle.tet_energy(x, T, rBm, rW, MU, LAM)
    assert np.allclose(psi.cpu().numpy(), rpsi, rtol=2e-6, atol=1e-6 * np.abs(rpsi).max())
    assert e.item() == pytest.approx(float(psi.cpu().numpy().astype(np.float64).sum()), rel=1e-12)


def test_out_of_range_tets_write_zeros(dev):
    x = torch.zeros((4, 3), dtype=torch.float32, device=dev)
    x[1, 0] = x[2, 1] = x[3, 2] = 1.0
    T = torch.tensor([[0, 1, 2, 3], [0, 1, 2, 9]], dtype=torch.int32, device=dev)
    Bm, W = ops.tet_rest(x, T)
    rows = torch.full((32,), -1, dtype=torch.int32, device=dev)
    cols = torch.full((32,), -1, dtype=torch.int32, device=dev)
    vals = torch.full((32, 3, 3), float("nan"), dtype=torch.float32, device=dev)
    ops.tet_hessian(x, T, Bm, W, MU, LAM, rows, cols, vals)
    torch.cuda.synchronize()
    assert W[1].item() == 0.0 and (rows[16:] == 0).all() and (vals[16:] == 0).all()
    assert torch.isfinite(vals[:16]).all()


@pytest.mark.parametrize("n", [1, 31, 32, 33, 127, 128, 129, 1000])
def test_partial_workgroups_and_shared_vertices(dev, oracle, n):
    """Tet counts around a wave's 32 and a workgroup's 128, every tet on its
    own vertices, tets sharing four vertices, and tets 1024 vertices apart and
    more: blocks bit-exact, forces within the rounding of the float sums of at
    most n terms."""
    rng = np.random.default_rng(n)
    unit = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], np.float32)
    for kind in ("own", "shared", "apart"):
        nv = {"own": 4 * n, "shared": 4, "apart": 4096 * 4}[kind]
        xcs = (np.tile(unit, (nv // 4, 1)) + 0.1 * rng.normal(size=(nv, 3))).astype(np.float32)
        x = (xcs + 0.1 * rng.normal(size=xcs.shape)).astype(np.float32)
        first = {"own": 4 * np.arange(n), "shared": np.zeros(n, int), "apart": 1024 * rng.integers(0, 16, n)}[kind]
        T = (first[:, None] + np.arange(4)).astype(np.int32)
        xcs_t, x_t, T_t = (torch.from_numpy(a).to(dev) for a in (xcs, x, T))
        Bm, W = ops.tet_rest(xcs_t, T_t)
        rows = torch.empty(16 * n, dtype=torch.int32, device=dev)
        cols = torch.empty_like(rows)
        vals = torch.empty((16 * n, 3, 3), dtype=torch.float32, device=dev)
        b = torch.zeros_like(x_t)
        ops.tet_hessian(x_t, T_t, Bm, W, MU, LAM, rows, cols, vals, b)
        torch.cuda.synchronize()
        rBm, rW = oracle.tet_rest(xcs, T)
        rr, rc, rv, rf = oracle.tet_hessian(x, T, rBm, rW, MU, LAM)
        assert np.array_equal(rows.cpu().numpy(), rr) and np.array_equal(cols.cpu().numpy(), rc)
        assert np.array_equal(vals.cpu().numpy().view(np.uint32), rv.view(np.uint32))
        assert np.abs(b.cpu().numpy() - rf).max() <= max(n, 16) * 2.0 ** -23 * np.abs(rf).max()


@pytest.mark.parametrize("V,n", [(4, 1), (4, 33), (8, 32), (40, 32), (40, 131), (3000, 257)])
def test_forces_of_crowded_vertices(dev, oracle, V, n):
    """Forces summed per vertex over a wave's 32 tets: one tet, four vertices
    in all of them, runs across the chunks of 64, and hardly any shared."""
    rng = np.random.default_rng(V + n)
    xcs, x = rng.random((V, 3)).astype(np.float32), rng.random((V, 3)).astype(np.float32)
    T = np.stack([rng.permutation(V)[:4] for _ in range(n)]).astype(np.int32)
    xcs_t, x_t, T_t = (torch.from_numpy(a).to(dev) for a in (xcs, x, T))
    Bm, W = ops.tet_rest(xcs_t, T_t)
    rows = torch.empty(16 * n, dtype=torch.int32, device=dev)
    cols = torch.empty_like(rows)
    vals = torch.empty((16 * n, 3, 3), dtype=torch.float32, device=dev)
    b = torch.zeros_like(x_t)
    ops.tet_hessian(x_t, T_t, Bm, W, MU, LAM, rows, cols, vals, b)
    rBm, rW = oracle.tet_rest(xcs, T)
    f = [oracle.tet_hessian(x, T[e:e + 1], rBm[e:e + 1], rW[e:e + 1], MU, LAM)[3] for e in range(n)]
    # n terms at most a vertex, in any order
    bound = (n + 1) * 2.0 ** -24 * np.abs(np.asarray(f, np.float64)).sum(0).max()
    assert np.abs(b.cpu().numpy() - np.asarray(f, np.float64).sum(0)).max() <= bound


@pytest.mark.parametrize("scale", [1.0, 1e9, 1e13, 3e18, 3e19, 1e25, 3e37])
def test_overflowing_tets_match_oracle(dev, oracle, scale):
    """Positions up to the largest floats, single infinite and NaN coordinates,
    and rest shapes that are flat, tiny or huge: every block is the oracle's,
    and NaN where its dense products with zero are NaN; forces NaN where its
    are."""
    rng = np.random.default_rng(3)
    n = 256
    xcs = rng.random((n, 4, 3)).astype(np.float32)
    x = (rng.normal(size=(n, 4, 3)) * scale).astype(np.float32)
    xcs[:32, 3] = xcs[:32, 0]
    xcs[32:64, :, 2] = 0
    xcs[64:96] *= 1e-12
    xcs[96:128] *= 1e12
    x[100:140, :, 0] = 0
    for k, bad in ((140, np.inf), (160, -np.inf), (180, np.nan)):
        for e in range(k, k + 12):
            x[e, (e - k) // 3, (e - k) % 3] = bad
    xcs, x = xcs.reshape(-1, 3), x.reshape(-1, 3)
    T = np.arange(4 * n, dtype=np.int32).reshape(n, 4)
    xcs_t, x_t, T_t = (torch.from_numpy(a).to(dev) for a in (xcs, x, T))
    Bm, W = ops.tet_rest(xcs_t, T_t)
    rows = torch.empty(16 * n, dtype=torch.int32, device=dev)
    cols = torch.empty_like(rows)
    vals = torch.empty((16 * n, 3, 3), dtype=torch.float32, device=dev)
    b = torch.zeros_like(x_t)
    ops.tet_hessian(x_t, T_t, Bm, W, MU, LAM, rows, cols, vals, b)
    rBm, rW = oracle.tet_rest(xcs, T)
    _, _, rv, rf = oracle.tet_hessian(x, T, rBm, rW, MU, LAM)
    gv, gf = vals.cpu().numpy(), b.cpu().numpy()
    assert np.array_equal(np.isnan(gv), np.isnan(rv)) and np.array_equal(np.isnan(gf), np.isnan(rf))
    assert np.array_equal(gv, rv, equal_nan=True)


def _slot(v):
    """The slot of a wave's 256 that vertex v asks for first (two vertices a
    lane): force_sums.hpp's hash."""
    h = (v.astype(np.uint64) >> np.uint64(4)) * np.uint64(2654435761) & np.uint64(0xffffffff)
    return ((h >> np.uint64(12)) & np.uint64(240)) + ((v.astype(np.uint64) + (h >> np.uint64(28))) & np.uint64(15))


@pytest.mark.parametrize("slots", [(0,), (5,), (240,), (255,), (0, 15, 16, 240, 255)])
def test_forces_of_colliding_vertices(dev, oracle, slots):
    """Strips of tets (each shares a vertex with the one before, so that a wave
    sums) whose 97 vertices a wave all ask for the same slot of its 256, the
    first, the last and the last group's among them: every search walks the
    others' slots, past the last group too. Each vertex is in two tets at
    most."""
    rng = np.random.default_rng(slots[0])
    n = 32 * 5 + 9
    ids = np.arange(16 * 40000)
    ids = rng.permutation(ids[np.isin(_slot(ids), slots)])
    assert ids.size >= 3 * n + 1
    T = ids[3 * np.arange(n)[:, None] + np.arange(4)].astype(np.int32)
    nv = int(T.max()) + 1
    xcs, x = (rng.normal(size=(nv, 3)).astype(np.float32) for _ in range(2))
    xcs_t, x_t, T_t = (torch.from_numpy(a).to(dev) for a in (xcs, x, T))
    Bm, W = ops.tet_rest(xcs_t, T_t)
    rows = torch.empty(16 * n, dtype=torch.int32, device=dev)
    cols = torch.empty_like(rows)
    vals = torch.empty((16 * n, 3, 3), dtype=torch.float32, device=dev)
    b = torch.zeros_like(x_t)
    ops.tet_hessian(x_t, T_t, Bm, W, MU, LAM, rows, cols, vals, b)
    rBm, rW = oracle.tet_rest(xcs, T)
    f = np.zeros((2, nv, 3))
    for e in range(n):
        one = oracle.tet_hessian(x[T[e]], np.arange(4, dtype=np.int32)[None], rBm[e:e + 1], rW[e:e + 1], MU, LAM)[3]
        f[0, T[e]] += one
        f[1, T[e]] += np.abs(one)
    assert (np.abs(b.cpu().numpy() - f[0]) <= 3 * 2.0 ** -24 * f[1]).all()
