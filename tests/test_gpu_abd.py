"""GPU affine-body contact reduction (affine_body_dynamics.py:144-190)
against the oracle's fp64 restatement, on the contact Hessian of the
64-icosphere grid (one body fixed) and of the screw in its fixed nut.

Bars: the DOF-level pattern (offsets, columns) exact; every value within
1e-5 of the sum of the absolute values of its terms plus fp32 rounding of the
result, and the reduced force within 1e-5 of its largest entry. (The sums are
fp64: the tests that say so hold them to one fp32 rounding.)"""
import numpy as np
import pytest
import torch

from ipc_warp_amd import scenes
from ipc_warp_amd.abd import AbdReducer
from ipc_warp_amd.contact import ContactSolverBase

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


def _case(dev, name):
    if name == "grid":
        soup, _ = scenes.icosphere_grid(seed=0)
        fixed = np.zeros(soup.n_bodies, np.int32)
        fixed[5] = 1
    else:
        soup = scenes.screw_and_nut(seed=0)[0]
        fixed = np.array([0, 1], np.int32)
    x = torch.from_numpy(soup.x).to(dev)
    S = ContactSolverBase(x, x.clone(), torch.from_numpy(soup.edges), torch.from_numpy(soup.triangles),
                          torch.from_numpy(soup.body), thickness=5e-4, buffer_=5e-4, kappa=1e8,
                          disable_self_collision_=True)
    S.detect_collision()
    b = torch.zeros_like(x)
    trip = S.compute_collision_hessian(b)
    # rest-frame coordinates: vertex minus its body's mean
    nb = int(soup.body.max()) + 1
    cen = np.zeros((nb, 3))
    np.add.at(cen, soup.body, soup.x.astype(np.float64))
    cen /= np.bincount(soup.body, minlength=nb)[:, None]
    rest = (soup.x - cen[soup.body]).astype(np.float32)
    return soup, nb, fixed, rest, trip, b, S


@pytest.mark.parametrize("name", ["grid", "screw"])
def test_reduction_matches_oracle(dev, oracle, name):
    soup, nb, fixed, rest, trip, b, S = _case(dev, name)
    _say(f"abd [{name}] bodies={nb} triplets={trip.rows.shape[0]}")
    scale = 1e-4
    R = AbdReducer()
    M, rf = R.reduce(nb, torch.from_numpy(soup.body).to(dev), torch.from_numpy(rest).to(dev),
                     torch.from_numpy(fixed).to(dev), trip.rows, trip.cols, trip.vals, b, scale)
    torch.cuda.synchronize()
    rows, cols, vals = trip.rows.cpu().numpy(), trip.cols.cpu().numpy(), trip.vals.cpu().numpy()
    o, c, v, a, rref = oracle.abd_reduce(nb, soup.body, rest, fixed, rows, cols, vals, b.cpu().numpy(), scale)
    nnz = int(o[-1])
    assert nnz > 0
    assert np.array_equal(M.offsets.cpu().numpy(), o)
    assert np.array_equal(M.columns[:nnz].cpu().numpy(), c)
    g = M.values[:nnz].cpu().numpy().astype(np.float64)
    err = np.abs(g - v)
    bound = 1e-5 * a + 6e-8 * np.abs(v) + 1e-30
    assert (err <= bound).all(), f"worst {float((err / bound).max())}"
    assert np.abs(rf.cpu().numpy() - rref).max() <= 1e-5 * np.abs(rref).max()
    # a second call on the same workspace gives the same pattern
    M2, _ = R.reduce(nb, torch.from_numpy(soup.body).to(dev), torch.from_numpy(rest).to(dev),
                     torch.from_numpy(fixed).to(dev), trip.rows, trip.cols, trip.vals, None, scale)
    assert torch.equal(M2.offsets, M.offsets)
    assert np.abs(M2.values[:nnz].cpu().numpy() - g).max() <= 1e-5 * a.max()


def test_capacity_is_reported_before_any_output(dev, oracle):
    from ipc_warp_amd._lib import lib

    soup, nb, fixed, rest, trip, b, S = _case(dev, "grid")
    R = AbdReducer()
    offsets = torch.empty(4 * nb + 1, dtype=torch.int32, device=dev)
    rf = torch.zeros((4 * nb, 3), dtype=torch.float32, device=dev)
    body_t = torch.from_numpy(soup.body).to(dev)
    rest_t = torch.from_numpy(rest).to(dev)
    fixed_t = torch.from_numpy(fixed).to(dev)
    st = lib().ipc_abd_reduce_contacts(R.handle, nb, body_t.data_ptr(), rest_t.data_ptr(), fixed_t.data_ptr(),
                                       soup.x.shape[0], trip.rows.data_ptr(), trip.cols.data_ptr(),
                                       trip.vals.data_ptr(), trip.rows.shape[0], b.data_ptr(), 1.0,
                                       offsets.data_ptr(), None, None, 0, rf.data_ptr(), None)
    torch.cuda.synchronize()
    assert st > 0 and st % 16 == 0 and int(offsets[-1].item()) == st
    assert not rf.any()


@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 70001])
@pytest.mark.parametrize("nb", [1, 3, 40])
def test_queue_edges_match_oracle(dev, oracle, n, nb):
    """Triplet counts around a tile of the reduction's queue (1024), bodies
    that change from lane to lane, zero blocks, vertices out of range, a fixed
    body, and more body pairs than the mark kernel's LDS set holds (40^2);
    the reduction's bars."""
    rng = np.random.default_rng(n + nb)
    nv = 500
    body = np.sort(rng.integers(0, nb, nv)).astype(np.int32)
    fixed = np.zeros(nb, np.int32)
    if nb > 1:
        fixed[nb // 2] = 1
    rest = rng.normal(size=(nv, 3)).astype(np.float32)
    rows, cols = rng.integers(-1, nv + 1, (2, n)).astype(np.int32)
    vals = rng.normal(size=(n, 3, 3)).astype(np.float32)
    vals[rng.random(n) < 0.3] = 0.0
    force = rng.normal(size=(nv, 3)).astype(np.float32)
    M, rf = AbdReducer().reduce(nb, *(torch.from_numpy(a).to(dev) for a in (body, rest, fixed, rows, cols, vals, force)),
                                scale=0.5)
    o, c, v, a, rref = oracle.abd_reduce(nb, body, rest, fixed, rows, cols, vals, force, 0.5)
    nnz = int(o[-1])
    assert np.array_equal(M.offsets.cpu().numpy(), o)
    assert np.array_equal(M.columns[:nnz].cpu().numpy(), c)
    err = np.abs(M.values[:nnz].cpu().numpy().astype(np.float64) - v)
    assert (err <= 1e-5 * a + 6e-8 * np.abs(v) + 1e-30).all()
    assert np.abs(rf.cpu().numpy() - rref).max() <= 1e-5 * max(np.abs(rref).max(), 1e-30)


def _reduce(dev, nb, body, rest, rows, cols, vals, force):
    fixed = np.zeros(nb, np.int32)
    M, rf = AbdReducer().reduce(nb, *(torch.from_numpy(np.ascontiguousarray(a)).to(dev)
                                      for a in (body, rest, fixed, rows, cols, vals, force)), scale=1.0)
    torch.cuda.synchronize()
    return M, rf.cpu().numpy().reshape(-1, 3)


@pytest.mark.parametrize("n", [1, 63, 513, 4096, 118000])
@pytest.mark.parametrize("nb", [1, 3, 40, 1000])
def test_forces_are_summed_in_double(dev, n, nb):
    """Forces whose sums fp32 partial sums lose (ones beside 2^24, and random
    ones that nearly cancel), of bodies from one vertex to runs of many waves:
    the fp64 sum rounded once to fp32. fp64 sums of n terms, here and in the
    oracle, are off by n 2^-53 of the magnitudes' sum."""
    rng = np.random.default_rng(n + nb)
    body = np.sort(rng.integers(0, nb, n)).astype(np.int32)
    rest = rng.normal(size=(n, 3)).astype(np.float32)
    none = np.zeros(1, np.int32)
    big = np.ones((n, 3), np.float32)
    big[:: 64 * 3] = 2.0 ** 24
    for force in (big, rng.normal(size=(n, 3)).astype(np.float32)):
        _, rf = _reduce(dev, nb, body, rest, none, none, np.zeros((1, 3, 3), np.float32), force)
        c = np.concatenate([np.ones((n, 1)), rest.astype(np.float64)], 1)
        t = (c[:, :, None] * force.astype(np.float64)[:, None, :]).reshape(n, 12)
        want, mag = np.zeros((nb, 12)), np.zeros((nb, 12))
        np.add.at(want, body, t)
        np.add.at(mag, body, np.abs(t))
        err = np.abs(rf.reshape(nb, 12) - want)
        assert (err <= 2.0 ** -24 * np.abs(want) + 2 * n * 2.0 ** -53 * mag).all()


@pytest.mark.parametrize("n", [1, 63, 1025, 70001, 1000003])
@pytest.mark.parametrize("nb", [1, 3])
def test_blocks_are_summed_in_double(dev, oracle, n, nb):
    """Blocks that a lane adds many of to the same body pair: the fp64 sum
    rounded once to fp32. fp64 sums of n terms, here and in the oracle, are off
    by n 2^-53 of the magnitudes' sum, and a term by its two products."""
    rng = np.random.default_rng(n + nb)
    nv = 300
    body = np.sort(rng.integers(0, nb, nv)).astype(np.int32)
    rest = rng.normal(size=(nv, 3)).astype(np.float32)
    rows, cols = np.sort(rng.integers(0, nv, (2, n)), axis=1).astype(np.int32)
    vals = rng.normal(size=(n, 3, 3)).astype(np.float32)
    vals[:: 64 * 3] = 2.0 ** 24
    M, _ = _reduce(dev, nb, body, rest, rows, cols, vals, np.zeros((nv, 3), np.float32))
    o, c, v, a, _ = oracle.abd_reduce(nb, body, rest, np.zeros(nb, np.int32), rows, cols, vals, None, 1.0)
    nnz = int(o[-1])
    assert np.array_equal(M.offsets.cpu().numpy(), o)
    assert np.array_equal(M.columns[:nnz].cpu().numpy(), c)
    err = np.abs(M.values[:nnz].cpu().numpy().astype(np.float64) - v)
    assert (err <= 2.0 ** -24 * np.abs(v) + 2 * (n + 4) * 2.0 ** -53 * a).all()


@pytest.mark.parametrize("n", [2048 * 64, 2048 * 64 + 1, 2048 * 960 + 1, 2048 * 1024 + 1])
def test_run_edges_match_oracle(dev, oracle, n):
    """Triplet counts around the changes of a workgroup's run (64 more, then
    whole tiles of 1024), with 12^2 body pairs in turn; the bars of the fp64
    sums."""
    rng = np.random.default_rng(n)
    nv, nb = 600, 12
    body = np.sort(rng.integers(0, nb, nv)).astype(np.int32)
    rest = rng.normal(size=(nv, 3)).astype(np.float32)
    quads = rng.integers(0, nv, (n // 16 + 1, 4)).astype(np.int32)
    rows, cols = np.repeat(quads, 4, 1).reshape(-1)[:n], np.tile(quads, (1, 4)).reshape(-1)[:n]
    vals = rng.normal(size=(n, 3, 3)).astype(np.float32)
    M, _ = _reduce(dev, nb, body, rest, rows, cols, vals, np.zeros((nv, 3), np.float32))
    o, c, v, a, _ = oracle.abd_reduce(nb, body, rest, np.zeros(nb, np.int32), rows, cols, vals, None, 1.0)
    nnz = int(o[-1])
    assert np.array_equal(M.offsets.cpu().numpy(), o)
    assert np.array_equal(M.columns[:nnz].cpu().numpy(), c)
    err = np.abs(M.values[:nnz].cpu().numpy().astype(np.float64) - v)
    assert (err <= 2.0 ** -24 * np.abs(v) + 2 * (n + 4) * 2.0 ** -53 * a).all()


@pytest.mark.parametrize("partners", [1, 2, 4, 5, 6, 30])
def test_flush_batches_match_oracle(dev, oracle, partners):
    """Waves that hand over one body pair, up to five in a batch and more than
    five, with lanes that hold nothing among them: contacts of one body with 1
    to 30 others, in turn and in runs; the bars of the fp64 sums."""
    rng = np.random.default_rng(partners)
    nb, per, k = 64, 9, 9000
    body = np.repeat(np.arange(nb), per).astype(np.int32)
    nv = nb * per
    rest = rng.normal(size=(nv, 3)).astype(np.float32)
    a = np.sort(rng.integers(0, nb, k))
    b = (a + np.where(np.arange(k) < k // 2, np.arange(k) % partners, rng.integers(0, partners, k))) % nb
    quads = np.stack([a * per + rng.integers(0, per, k), a * per + rng.integers(0, per, k),
                      b * per + rng.integers(0, per, k), b * per + rng.integers(0, per, k)], 1).astype(np.int32)
    rows, cols = np.repeat(quads, 4, 1).reshape(-1), np.tile(quads, (1, 4)).reshape(-1)
    n = rows.size
    vals = rng.normal(size=(n, 3, 3)).astype(np.float32)
    vals[rng.random(n) < 0.4] = 0.0
    M, _ = _reduce(dev, nb, body, rest, rows, cols, vals, np.zeros((nv, 3), np.float32))
    o, c, v, s, _ = oracle.abd_reduce(nb, body, rest, np.zeros(nb, np.int32), rows, cols, vals, None, 1.0)
    nnz = int(o[-1])
    assert np.array_equal(M.offsets.cpu().numpy(), o)
    assert np.array_equal(M.columns[:nnz].cpu().numpy(), c)
    err = np.abs(M.values[:nnz].cpu().numpy().astype(np.float64) - v)
    assert (err <= 2.0 ** -24 * np.abs(v) + 2 * (n + 4) * 2.0 ** -53 * s).all()
