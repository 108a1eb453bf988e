"""The particle layer on the GPU (pfs_particles_advect, pfs_ngrid_*,
pfs_scan_exclusive_u32) against its CPU oracle: integer outputs and
positions bit-exact, densities bit-exact (same summation order)."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import particles as op  # noqa: E402
from probabilistic_fluid_simulation_amd import particles, scenes  # noqa: E402
from probabilistic_fluid_simulation_amd.fluid import VPField  # noqa: E402

pytestmark = pytest.mark.gpu


def _u32(t: torch.Tensor) -> np.ndarray:
    return t.cpu().numpy().view(np.uint32)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1000, 4095, 4096, 4097, 70000, 1 << 20])
def test_scan_exclusive(n):
    rng = np.random.default_rng(n)
    a = rng.integers(0, 50, size=n).astype(np.int32)
    out, total = particles.scan_exclusive(torch.from_numpy(a).cuda())
    want = np.zeros(n, np.int64)
    want[1:] = np.cumsum(a, dtype=np.int64)[:-1]
    np.testing.assert_array_equal(out.cpu().numpy().astype(np.int64), want)
    assert total == int(a.sum())


@pytest.mark.parametrize("n", [4096 * 8 - 1, 4096 * 8, 4096 * 8 + 1])
def test_scan_in_one_and_two_launches(n):
    test_scan_exclusive(n)


@pytest.mark.parametrize("n", [4096, 4097, 8192, 4096 * 8, 4096 * 8 + 1])
def test_scan_in_place(n):
    """out == in: one block, blocks that may not read what others write, and
    the count past which totals have a launch of their own anyway."""
    from probabilistic_fluid_simulation_amd import _lib

    a = np.random.default_rng(n).integers(0, 50, size=n).astype(np.int32)
    t = torch.from_numpy(a).cuda()
    total = torch.zeros(1, dtype=torch.int32, device="cuda")
    ws = torch.empty((n + 4095) // 4096 + 1, dtype=torch.int32, device="cuda")
    _lib.call("pfs_scan_exclusive_u32", t.data_ptr(), t.data_ptr(), n, total.data_ptr(),
              ws.data_ptr(), ws.numel() * 4, torch.cuda.current_stream().cuda_stream)
    np.testing.assert_array_equal(t.cpu().numpy(), np.cumsum(a) - a)
    assert int(total.item()) == int(a.sum())


def _positions(n, W, H, seed):
    rng = np.random.default_rng(seed)
    x = np.minimum((rng.random(n) * W).astype(np.float32), np.nextafter(np.float32(W), np.float32(0)))
    y = np.minimum((rng.random(n) * H).astype(np.float32), np.nextafter(np.float32(H), np.float32(0)))
    return x, y


def _check_grid(x, y, W, H, r, mass=1.0):
    n = len(x)
    ng = particles.NeighborGrid(n, W, H, r)
    ng.build(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda())
    og = op.Grid(x, y, W, H, r, ng.g.gx, ng.g.gy, ng.g.kx, ng.g.ky)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(_u32(ng.keys), og.keys)
    np.testing.assert_array_equal(_u32(ng.order), og.order)
    np.testing.assert_array_equal(_u32(ng.cell_start), og.start)
    np.testing.assert_array_equal(_u32(ng.cell_end), og.end)
    assert ng.xs.cpu().numpy().tobytes() == og.xs.tobytes()
    assert ng.ys.cpu().numpy().tobytes() == og.ys.tobytes()
    counts, offsets, nbr = ng.neighbors()
    oc, oo, on = og.neighbors()
    np.testing.assert_array_equal(_u32(counts), oc)
    np.testing.assert_array_equal(_u32(offsets), oo)
    np.testing.assert_array_equal(_u32(nbr), on)
    rho = ng.density(mass)
    assert rho.cpu().numpy().tobytes() == og.density(mass).tobytes()
    rho2, c2 = ng.density(mass, with_counts=True)
    assert rho2.cpu().numpy().tobytes() == og.density(mass).tobytes()
    np.testing.assert_array_equal(_u32(c2), oc)
    return ng


# cell counts spanning every radix plan: 1 pass (< 2^8 cells), 2 x 8 bits,
# 2 x 10 bits (150K cells), 3 x 8 bits (1.2M cells), 3 x 10 bits (17.6M cells)
@pytest.mark.parametrize("n,W,H,r", [(1, 16.0, 16.0, 1.0), (777, 40.0, 30.0, 2.5),
                                     (5000, 100.0, 100.0, 1.5), (9000, 500.0, 300.0, 1.0),
                                     (4097, 64.0, 64.0, 3.9), (600, 20.0, 13.0, 3.9),
                                     (3000, 1100.0, 1100.0, 1.0), (3000, 4200.0, 4200.0, 1.0)])
def test_grid_and_neighbors_match_oracle(n, W, H, r):
    x, y = _positions(n, W, H, seed=n)
    _check_grid(x, y, W, H, r)


def test_lists_and_density_across_the_wrap_at_a_corner():
    """600 particles within 3 of a corner of a 4096 x 4096 domain (r = 1.5):
    every list crosses the wrap in x, y or both, from either side, which
    takes every per-range shift of the edge traversal."""
    rng = np.random.default_rng(5)
    W = 4096.0
    x = ((rng.random(600) * 6 - 3) % W).astype(np.float32)
    y = ((rng.random(600) * 6 - 3) % W).astype(np.float32)
    x[x >= np.float32(W)] = 0
    y[y >= np.float32(W)] = 0
    ng = _check_grid(x, y, W, W, 1.5)
    assert ng.g.gx >= 7


@pytest.mark.parametrize("n", [(1 << 18) - 1, 1 << 18, (1 << 18) + 65])
def test_either_side_of_the_lane_rule(n):
    """Four lanes a particle below 2^18 particles, one from there on (counts
    and density): domain edges on all sides."""
    x, y = _positions(n, 420.0, 300.0, seed=n)
    _check_grid(x, y, 420.0, 300.0, 1.4)


@pytest.mark.parametrize("n,W,H", [
    (16 << 10, 90.0, 70.0), ((16 << 10) + 1, 90.0, 70.0),    # 8-bit digits, 16 / 17 tiles
    (16 << 11, 500.0, 300.0), ((16 << 11) + 1, 500.0, 300.0),  # 10-bit
    (1 << 19, 90.0, 70.0), ((1 << 19) + 1, 90.0, 70.0),      # small and large tiles
    (1 << 19, 500.0, 300.0), ((1 << 19) + 1, 500.0, 300.0),
    ((1 << 22) + 1, 500.0, 300.0)])                          # 1025 tiles a row
def test_grid_at_the_edges_of_the_sorts_tiles(n, W, H):
    """Keys, order and cell tables against a stable argsort; a third of the
    particles lie in one cell, so that its table's neighbours are far apart."""
    x, y = _positions(n, W, H, seed=n)
    x[::3], y[::3] = 40.25, 50.75
    ng = particles.NeighborGrid(n, W, H, 1.0)
    ng.build(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda())
    g = ng.g
    cx = np.minimum((x * np.float32(g.kx)).astype(np.int64), g.gx - 1)
    cy = np.minimum((y * np.float32(g.ky)).astype(np.int64), g.gy - 1)
    key = cy * g.gx + cx
    order = np.argsort(key, kind="stable")
    np.testing.assert_array_equal(_u32(ng.keys), key)
    np.testing.assert_array_equal(_u32(ng.order), order)
    cells = np.arange(g.gx * g.gy)
    np.testing.assert_array_equal(_u32(ng.cell_start), np.searchsorted(key[order], cells))
    np.testing.assert_array_equal(_u32(ng.cell_end), np.searchsorted(key[order], cells, "right"))
    np.testing.assert_array_equal(ng.xs.cpu().numpy(), x[order])
    np.testing.assert_array_equal(ng.ys.cpu().numpy(), y[order])


@pytest.mark.parametrize("n", [(1 << 16) - 3, 1 << 16, (1 << 16) + 1])
@pytest.mark.parametrize("r", [1.4, 3.1], ids=["short-rows", "long-rows"])
def test_either_side_of_the_list_lanes(n, r):
    """16 lanes a particle up to 2^16 (counts and lists, by id and by sorted
    position), four above."""
    x, y = _positions(n, 220.0, 160.0, seed=n)
    ng = _check_grid(x, y, 220.0, 160.0, r)
    og = op.Grid(x, y, 220.0, 160.0, r, ng.g.gx, ng.g.gy, ng.g.kx, ng.g.ky)
    got, want = ng.neighbors(by_position=True), og.neighbors(by_position=True)
    for t, w in zip(got, want):
        np.testing.assert_array_equal(_u32(t), w)


def test_clustered_particles_and_empty_cells():
    """Many particles in few cells (long equal-key runs across sort tiles)."""
    rng = np.random.default_rng(11)
    n = 20000
    x = (10.0 + rng.random(n) * 3.0).astype(np.float32)
    y = (20.0 + rng.random(n) * 2.0).astype(np.float32)
    _check_grid(x, y, 64.0, 64.0, 1.0)


@pytest.mark.parametrize("w,h", [(64, 64), (50, 38)])
def test_tracer_advect_matches_oracle(w, h):
    s = scenes.random_scene(w, h, w, h, seed=w, dt=0.7, visc=0.1, iters=4)
    x, y = scenes.particles_disk(3000, w, h, seed=w)
    xg, yg = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    vp = VPField.from_numpy(s.vp)
    xo, yo = x.copy(), y.copy()
    for _ in range(10):
        particles.advect(xg, yg, vp, s.dt)
        op.advect(xo, yo, s.vp, s.dt)
    assert xg.cpu().numpy().tobytes() == xo.tobytes()
    assert yg.cpu().numpy().tobytes() == yo.tobytes()


def test_16k_workload_steps():
    """The 16K particle workload: tracers through the evolving 128x128 field
    (the GPU step), the grid rebuilt every step, checked against the oracle
    fed the same field each step."""
    from probabilistic_fluid_simulation_amd import fluid

    s, x, y, r = scenes.particles_16k()
    vp, tmp = VPField.from_numpy(s.vp), VPField.from_numpy(s.tmp)
    xg, yg = torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda()
    xo, yo = x.copy(), y.copy()
    for _ in range(5):
        fluid.simulate_fluid_step(vp, tmp, s.dt, s.visc, s.iters)
        particles.advect(xg, yg, vp, s.dt)
        op.advect(xo, yo, vp.numpy(), s.dt)
    assert xg.cpu().numpy().tobytes() == xo.tobytes()
    _check_grid(xo, yo, 128.0, 128.0, r, mass=1.0 / len(x))


def test_errors():
    with pytest.raises(Exception):
        particles.NeighborGrid(10, 4.0, 4.0, 2.0)
    ng = particles.NeighborGrid(10, 16.0, 16.0, 1.0)
    x = torch.zeros(11, device="cuda")
    with pytest.raises(ValueError):
        ng.build(x, x)


def test_tracers_kept_in_cell_order_match_oracle():
    """Tracers that adopt the sort every step: positions, ids, tables, lists
    (by sorted position) and densities against the oracle doing the same."""
    s = scenes.random_scene(96, 80, 96, 80, seed=21, dt=0.8, visc=0.1, iters=4)
    x, y = scenes.particles_disk(6000, 96, 80, seed=21)
    vp = VPField.from_numpy(s.vp)
    tr = particles.Tracers(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda(), 96.0, 80.0, 1.5)
    g = tr.grid.g
    xo, yo, ids = x.copy(), y.copy(), np.arange(len(x), dtype=np.uint32)
    for step in range(4):
        tr.advect(vp, s.dt)
        tr.sort()
        op.advect(xo, yo, s.vp, s.dt)
        og = op.Grid(xo, yo, 96.0, 80.0, 1.5, g.gx, g.gy, g.kx, g.ky)
        xo, yo, ids = og.xs.copy(), og.ys.copy(), ids[og.order]
        assert tr.x.cpu().numpy().tobytes() == xo.tobytes(), step
        np.testing.assert_array_equal(_u32(tr.ids), ids)
        np.testing.assert_array_equal(_u32(tr.grid.order), og.order)
        np.testing.assert_array_equal(_u32(tr.grid.cell_start), og.start)
    counts, offsets, nbr = tr.neighbors()
    oc, oo, on = og.neighbors(by_position=True)
    np.testing.assert_array_equal(_u32(counts), oc)
    np.testing.assert_array_equal(_u32(offsets), oo)
    np.testing.assert_array_equal(_u32(nbr), on)
    assert tr.density(0.5).cpu().numpy().tobytes() == og.density(0.5, by_position=True).tobytes()


# ---------------------------------------------------------------- PBF solve
def _pbf_setup(n, W, h, seed, spread):
    rng = np.random.default_rng(seed)
    x = (W / 2 + rng.normal(0, spread, n)).astype(np.float32) % np.float32(W)
    y = (W / 2 + rng.normal(0, spread, n)).astype(np.float32) % np.float32(W)
    ng = particles.NeighborGrid(n, W, W, h)
    ng.build(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda())
    og = op.Grid(x, y, W, W, h, ng.g.gx, ng.g.gy, ng.g.kx, ng.g.ky)
    rho0 = float(np.median(og.density(1.0, by_position=True)))
    return ng, og, rho0


@pytest.mark.parametrize("iters,stop", [(0, None), (1, None), (6, None), (8, 3), (8, 2)],
                         ids=["0", "1", "6", "stop-at-3", "stop-at-2"])
def test_pbf_matches_oracle(iters, stop):
    """Positions and lambdas bit-exact to the oracle; the FP64 residuals
    equal to rounding (block sums on the GPU); the same iterate stops it."""
    ng, og, rho0 = _pbf_setup(5000, 40.0, 1.0, 11, 3.0)
    eps = 50.0
    tol = 0.0
    if stop is not None:
        _, _, _, res_all, _ = og.pbf(1.0, rho0, eps, iters)
        tol = float(np.sqrt((res_all[stop - 1] + res_all[stop]) / 2 / og.n))
    ox, oy, olam, ores, oused = og.pbf(1.0, rho0, eps, iters, tol)
    lam, res, used = ng.pbf(1.0, rho0, eps, iters, tol)
    torch.cuda.synchronize()
    assert int(used.item()) == oused == (iters if stop is None else stop)
    assert ng.xs.cpu().numpy().tobytes() == ox.tobytes()
    assert ng.ys.cpu().numpy().tobytes() == oy.tobytes()
    assert lam.cpu().numpy().tobytes() == olam.tobytes()
    r = res.cpu().numpy()
    done = ores >= 0
    np.testing.assert_array_equal(r >= 0, done)
    np.testing.assert_allclose(r[done], ores[done], rtol=1e-12)


@pytest.mark.parametrize("stop", [1, 2])
@pytest.mark.parametrize("n", [200001, 3 << 17], ids=["four-lanes", "one-lane"])
def test_pbf_converges_in_the_middle_of_a_launch(n, stop):
    """An iterate found converged while workgroups of the launch that records it
    are still to start (782 workgroups of 1024 threads, where 512 run at once),
    at an odd and an even iterate: the buffers and the residuals are those of
    a solve of that many iterations, and nothing follows it."""
    ng, og, rho0 = _pbf_setup(n, 1000.0, 1.5, 19, 130.0)
    _, _, _, res_all, _ = og.pbf(1.0, rho0, 5.0, 3)
    tol = float(np.sqrt((res_all[stop - 1] + res_all[stop]) / 2 / og.n))
    ox, oy, olam, ores, oused = og.pbf(1.0, rho0, 5.0, 4, tol)
    lam, res, used = ng.pbf(1.0, rho0, 5.0, 4, tol)
    assert int(used.item()) == oused == stop
    assert ng.xs.cpu().numpy().tobytes() == ox.tobytes()
    assert ng.ys.cpu().numpy().tobytes() == oy.tobytes()
    assert lam.cpu().numpy().tobytes() == olam.tobytes()
    r = res.cpu().numpy()
    np.testing.assert_allclose(r[:stop + 1], ores[:stop + 1], rtol=1e-12)
    assert (r[stop + 1:] == -1).all()


@pytest.mark.parametrize("n", [(3 << 17) - 1, 3 << 17])
def test_pbf_either_side_of_the_lane_rule(n):
    ng, og, rho0 = _pbf_setup(n, 1000.0, 1.5, 13, 130.0)
    ox, oy, olam, ores, _ = og.pbf(1.0, rho0, 5.0, 2)
    lam, res, _ = ng.pbf(1.0, rho0, 5.0, 2)
    torch.cuda.synchronize()
    assert ng.xs.cpu().numpy().tobytes() == ox.tobytes()
    assert ng.ys.cpu().numpy().tobytes() == oy.tobytes()
    assert lam.cpu().numpy().tobytes() == olam.tobytes()
    np.testing.assert_allclose(res.cpu().numpy(), ores, rtol=1e-12)


@pytest.mark.parametrize("scale", [1.0, 1e4], ids=["short-division", "plain-division"])
@pytest.mark.parametrize("n", [4000, 3 << 17])
def test_pbf_every_division(n, scale):
    """Radii inside and outside the short root and division's range, distances
    whose square's significand it excludes (1 - 2^-24 and its square), and
    pairs across the wrap in only some wavefronts."""
    rng = np.random.default_rng(17)
    W = np.float32((400.0 if n > 10000 else 40.0) * scale)
    x, y = ((rng.random(n) * W).astype(np.float32) for _ in range(2))
    x[x >= W] = 0
    y[y >= W] = 0
    x[:40], x[40:80] = 0.0, np.float32(scale) * np.float32(1 - 2.0 ** -24)
    y[40:80] = y[:40]
    r = 1.5 * scale
    ng = particles.NeighborGrid(n, float(W), float(W), r)
    ng.build(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda())
    og = op.Grid(x, y, float(W), float(W), r, ng.g.gx, ng.g.gy, ng.g.kx, ng.g.ky)
    rho0 = float(np.median(og.density(1.0, by_position=True)))
    ox, oy, olam, ores, _ = og.pbf(1.0, rho0, 5.0, 2)
    lam, res, _ = ng.pbf(1.0, rho0, 5.0, 2)
    assert ng.xs.cpu().numpy().tobytes() == ox.tobytes()
    assert ng.ys.cpu().numpy().tobytes() == oy.tobytes()
    assert lam.cpu().numpy().tobytes() == olam.tobytes()
    np.testing.assert_allclose(res.cpu().numpy(), ores, rtol=1e-12)


def test_pbf_on_tracers_and_errors():
    """Tracers.pbf works on the tracers' own (cell-ordered) positions; bad
    arguments are rejected before anything runs."""
    s, x, y, r = scenes.particles_16k()
    H, W = s.vp.shape[:2]
    tr = particles.Tracers(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda(), float(W),
                           float(H), r)
    tr.sort()
    rho = tr.density(1.0)
    rho0 = float(rho.median().item())
    og = op.Grid(tr.x.cpu().numpy(), tr.y.cpu().numpy(), float(W), float(H), r, tr.grid.g.gx,
                 tr.grid.g.gy, tr.grid.g.kx, tr.grid.g.ky)
    ox, oy, olam, ores, oused = og.pbf(1.0, rho0, 20.0, 4)
    lam, res, used = tr.pbf(1.0, rho0, 20.0, 4)
    torch.cuda.synchronize()
    assert tr.x.cpu().numpy().tobytes() == ox.tobytes()
    assert tr.y.cpu().numpy().tobytes() == oy.tobytes()
    assert np.all(np.diff(res.cpu().numpy()) < 0)
    from probabilistic_fluid_simulation_amd import _lib
    for bad in (dict(max_iters=65), dict(max_iters=-1)):
        with pytest.raises(ValueError):
            tr.pbf(1.0, rho0, 20.0, **bad)
    with pytest.raises(_lib.PfsError):
        tr.pbf(1.0, -1.0, 20.0, 2)


@pytest.mark.parametrize("n", [1, 3, 300])
def test_pbf_small_counts(n):
    """One particle (no neighbours), a few, and fewer than one workgroup."""
    ng, og, rho0 = _pbf_setup(n, 12.0, 1.0, 17, 0.8)
    ox, oy, olam, ores, oused = og.pbf(1.0, rho0, 10.0, 3)
    lam, res, used = ng.pbf(1.0, rho0, 10.0, 3)
    torch.cuda.synchronize()
    # one particle is its own rest density: sum C^2 = 0 <= tol^2 n stops at iterate 0
    assert int(used.item()) == oused == (0 if n == 1 else 3)
    assert ng.xs.cpu().numpy().tobytes() == ox.tobytes()
    assert ng.ys.cpu().numpy().tobytes() == oy.tobytes()
    assert lam.cpu().numpy().tobytes() == olam.tobytes()
    np.testing.assert_allclose(res.cpu().numpy(), ores, rtol=1e-12)


@pytest.mark.parametrize("order", [True, False], ids=["by-id", "by-position"])
def test_lists_from_density_counts(order):
    """pfs_ngrid_lists: lists from the density pass's counts equal those of
    pfs_ngrid_neighbors, for a fresh grid (buffer sized on the first call),
    a reused buffer, and one that must grow."""
    n, W = 6000, 40.0
    rng = np.random.default_rng(29)
    x = (W / 2 + rng.normal(0, 6.0, n)).astype(np.float32) % np.float32(W)
    y = (W / 2 + rng.normal(0, 6.0, n)).astype(np.float32) % np.float32(W)
    ng = particles.NeighborGrid(n, W, W, 1.0)
    ng.build(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda())
    og = op.Grid(x, y, W, W, 1.0, ng.g.gx, ng.g.gy, ng.g.kx, ng.g.ky)
    oc, oo, on = og.neighbors(by_position=not order)
    for _ in range(2):
        ng.density(1.0, by_position=not order, with_counts=True)
        counts, offsets, nbr = ng.neighbors(by_position=not order, counted=True)
        np.testing.assert_array_equal(_u32(counts), oc)
        np.testing.assert_array_equal(_u32(offsets), oo)
        np.testing.assert_array_equal(_u32(nbr), on)
    ng.nbr = ng.nbr[:10].clone()  # too small: grows
    ng.density(1.0, by_position=not order, with_counts=True)
    np.testing.assert_array_equal(_u32(ng.neighbors(by_position=not order, counted=True)[2]), on)
    assert ng.nbr.numel() >= len(on)


def test_sizes_of_work_on_another_stream():
    """A scan's total and the first lists' size are read after the stream they
    are made on, here busy for milliseconds, and not after the current one."""
    st = torch.cuda.Stream()
    m = torch.rand(8192, 8192, device="cuda")
    a = torch.ones(100000, dtype=torch.int32, device="cuda")
    x, y = (torch.from_numpy(p).cuda() for p in _positions(20000, 100.0, 100.0, seed=41))
    ng = particles.NeighborGrid(20000, 100.0, 100.0, 1.5)
    ng.build(x, y)
    torch.cuda.synchronize()
    with torch.cuda.stream(st):
        m @ m
    assert particles.scan_exclusive(a, stream=st)[1] == 100000
    with torch.cuda.stream(st):
        m @ m
    counts, _, nbr = ng.neighbors(stream=st)
    torch.cuda.synchronize()
    assert nbr.numel() == int(counts.sum().item()) > 0


@pytest.mark.parametrize("own_stream", [False, True], ids=["current-stream", "own-stream"])
@pytest.mark.parametrize("counted", [False, True], ids=["counting", "counted"])
def test_neighbors_returns_finished_lists(own_stream, counted):
    """Nothing is left queued when neighbors() returns, so that another stream
    reads whole lists: 1M particles of 37 neighbours, whose lists take far longer
    than the return."""
    n, W = 1 << 20, 512.0
    x, y = (torch.rand(n, device="cuda", generator=torch.Generator("cuda").manual_seed(s)) * 511.0
            for s in (31, 32))
    torch.cuda.synchronize()
    st = torch.cuda.Stream() if own_stream else torch.cuda.current_stream()
    ng = particles.NeighborGrid(n, W, W, 1.7)
    ng.build(x, y, st)
    for _ in range(3):
        ng.density(1.0, st, with_counts=True)
        ng.neighbors(st if own_stream else None, counted=counted)
        assert st.query()


@pytest.mark.parametrize("spread", [2.5, 4.0], ids=["dense", "sparse"])
def test_lists_by_position_bitexact(spread):
    """Lists by sorted position (written through LDS windows): a dense blob
    puts more entries in a wave's block than one window holds."""
    n, W = 20000, 40.0
    rng = np.random.default_rng(23)
    x = (W / 2 + rng.normal(0, spread * 4, n)).astype(np.float32) % np.float32(W)
    y = (W / 2 + rng.normal(0, spread * 4, n)).astype(np.float32) % np.float32(W)
    ng = particles.NeighborGrid(n, W, W, 1.0)
    ng.build(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda())
    og = op.Grid(x, y, W, W, 1.0, ng.g.gx, ng.g.gy, ng.g.kx, ng.g.ky)
    counts, offsets, nbr = ng.neighbors(by_position=True)
    oc, oo, on = og.neighbors(by_position=True)
    np.testing.assert_array_equal(_u32(counts), oc)
    np.testing.assert_array_equal(_u32(offsets), oo)
    np.testing.assert_array_equal(_u32(nbr), on)
    if spread < 3:
        per_wave = np.add.reduceat(oc.astype(np.int64), np.arange(0, n, 64))
        assert per_wave.max() > 2 * 3072  # three 3072-slot windows for some waves


def test_density_counts_with_a_non_finite_position():
    """A NaN position (its cell key clamps into the grid) is nobody's
    neighbour and has none itself: the density pass's counts equal the
    counting pass's (0 for it), and lists made from those counts equal the
    lists the counting pass makes."""
    x, y = _positions(3000, 100.0, 100.0, seed=77)
    x[17], y[17] = np.nan, np.nan
    x[1234] = np.inf
    ng = particles.NeighborGrid(len(x), 100.0, 100.0, 1.5)
    ng.build(torch.from_numpy(x).cuda(), torch.from_numpy(y).cuda())
    counts, offsets, nbr = (t.clone() for t in ng.neighbors())
    _, dcounts = ng.density(1.0, with_counts=True)
    dcounts = dcounts.clone()
    np.testing.assert_array_equal(_u32(dcounts), _u32(counts))
    assert _u32(counts)[17] == 0 and _u32(counts)[1234] == 0
    c2, o2, n2 = ng.neighbors(counted=True)
    np.testing.assert_array_equal(_u32(o2), _u32(offsets))
    np.testing.assert_array_equal(_u32(n2), _u32(nbr))
